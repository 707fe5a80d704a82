// Chunked forward of the gated delta rule, K = 256: the scan for launches that leave compute units idle, 16 columns of V to a workgroup
// and the keys split over two waves.
//
// The records, the stage and the reduction orders are those of the half-slice scan (gdn_chunk_scan32.h).  There a workgroup has 32 columns
// and a wave carries 16 of them through all 256 keys; a chunk takes what that wave needs to issue 108 MFMAs with everything around
// them.  With half of the CUs idle two waves share those 16 columns instead:
//     K S0, S0^T q^T, the decay, the update and the bf16 copies of the state are halved;
//     the halves of K S0 are added across the two waves through LDS, both form X and V~ (6 MFMAs);
//     the halves of S0^T q^T likewise, each wave finishing the output of 32 of the 64 tokens (4 MFMAs).
// 58 MFMAs a wave.  The waves hand over through an epoch word in LDS that the other polls (pair_publish, pair_wait): the products with q
// stand between writing the halves of K S0 and needing the other's.
//
// Bound by the instruction stream of a compute wave: the kernel over 30000 tokens, 3 heads, V = 512 (469 chunks) 808 us in half slices, 680
// here, 1.72 | 1.45 a chunk.  Forward, half slices | this: 64 tokens, 2 heads, V = 512 14.0 | 13.3 us, 777 tokens 36.1 | 33.1, 2000 68.7 |
// 60.3, 4 x 777 36.2 | 33.3.
// At K = 128, where 60 MFMAs become 34, what is duplicated and handed over eats what is saved: 4096 tokens, 16 heads, V = 128 87.0 | 88.8
// us.  And with 32 columns, four compute waves beside four loaders, it is slower for every size (777 tokens 37.2 | 38.0; 65536 tokens, 32
// heads, K = 128, V = 256 1572 | 1766).
//
// Counterpart upstream: fla's chunk_gated_delta_rule, reached from
// lm_engine/modeling_utils/sequence_mixer_blocks/gated_deltanet/module.py:197-209.

#include <type_traits>

#include "gdn_chunk32_common.h"
#include "gdn_launch.h"

namespace gdn {

namespace {

constexpr int K = 256;
constexpr int KEYS_WAVES = 8;  // 0 1 compute (a key half each) | 2 3 loaders | 4 output store | 5 exits at once | 6 7 loaders (as in the half-slice scan)
constexpr int KEYS_LOADERS = 4;

// Order of the MFMAs of one chunk in a compute wave ("ops"), and where its side work goes; placement is the earliest-deadline walk of
// Scan16Rules, at compile time:
//     K S0 (4 token tiles x K/64 slabs) | S0^T q^T (as many; the other wave's two tiles first) | V~ = T' X (6) | S += k^T V~' (2 K/32) |
//     O^T += V~^T P^T (this wave's two tiles x 2 slabs)
// "Logical" output tiles: 0 and 1 are this wave's, 2 and 3 the other's.
struct KeysRules {
    static constexpr int KW = K / 2;  // keys of a wave
    static constexpr int KS = KW / 32, KT = KW / 16;
    static constexpr int NS = 4 * KS, NQ = 4 * KS, NT = 6, NK = 2 * KT, NP = 4;
    static constexpr int OP_Q = NS, OP_T = OP_Q + NQ, OP_K = OP_T + NT, OP_P = OP_K + NK, NOPS = OP_P + NP;
    static constexpr int LA = 14;              // operand fragments are read this many ops ahead of their MFMA (726 us for 30000 tokens; 8 to 12 737)
    static constexpr int OP_BAR = NOPS - LA;   // the chunk's barrier: every read of its stage half has been issued
    static constexpr int AHEAD = 4, DIST = 3;  // scales are read AHEAD ops before their piece, results taken DIST ops after their MFMA

    // op j of the first two groups -> tile, key slab: two tiles alternate through all slabs, then the other two
    static constexpr int s_tile(int j) { return 2 * (j / (2 * KS)) + j % 2; }
    static constexpr int s_slab(int j) { return (j % (2 * KS)) / 2; }
    static constexpr int s_last(int t) { return (t / 2) * 2 * KS + 2 * (KS - 1) + t % 2; }
    static constexpr int q_tile(int j) { return (s_tile(j) + 2) % 4; }  // logical
    static constexpr int q_first(int l) { return ((l + 2) % 4 / 2) * 2 * KS + l % 2; }
    static constexpr int q_last(int l) { return s_last((l + 2) % 4); }
    // op j of T' X -> token tile, slab; fragment of the record (as in Scan16Rules)
    static constexpr int t_tile(int j) { return j < 4 ? j : j - 2; }
    static constexpr int t_slab(int j) { return j < 4 ? 0 : 1; }
    static constexpr int t_frag(int j) { return j < 2 ? j : j == 2 ? 2 : j == 3 ? 4 : j == 4 ? 3 : 5; }
    static constexpr int t_last(int t) { return t < 2 ? t : t + 2; }
    static constexpr int s_first(int s) { return s == 0 ? 0 : 4; }

    // The hand-overs: the halves of K S0 are published at OP_PUB_S and taken from OP_GET_S on, those of S0^T q^T at OP_PUB_Q and
    // OP_GET_Q.
    static constexpr int OP_PUB_S = OP_Q + DIST, OP_GET_S = OP_T - 2, OP_PUB_Q = OP_T + 4, OP_GET_Q = OP_K + 2;

    // pieces: half of K S0 of a token tile to the other wave | X of a token tile | X of a slab as operand | half of S0^T q^T of one of the
    // other wave's tiles to it | previous output tile to the staging | sum of both halves of an output tile, scaled | decay of a
    // state tile | scaled V~ of a token tile | plain V~ of a slab | new state slab
    static constexpr int N_SS = 4, N_XC = 4, N_XB = 2, N_QS = 2, N_OUT = 2, N_AS = 2, N_DEC = KT, N_VS = 4, N_VB = 2, N_SB = KS;
    static constexpr int P_SS = 0, P_XC = P_SS + N_SS, P_XB = P_XC + N_XC, P_QS = P_XB + N_XB, P_OUT = P_QS + N_QS, P_AS = P_OUT + N_OUT,
                         P_DEC = P_AS + N_AS, P_VS = P_DEC + N_DEC, P_VB = P_VS + N_VS, P_SB = P_VB + N_VB, NPIECES = P_SB + N_SB;
    struct Window {
        int first, end;  // the piece runs before the MFMA of an op in [first, end)
    };
    static constexpr int lesser(int a, int b) { return a < b ? a : b; }
    static constexpr Window window(int pc) {
        if (pc < P_XC) return {s_last(pc - P_SS) + DIST, OP_PUB_S + 1};  // (before the publishing in its op)
        if (pc < P_XB) return {OP_GET_S + 1, OP_T + s_first((pc - P_XC) / 2)};
        if (pc < P_QS) return {OP_GET_S + 1, OP_T + s_first(pc - P_XB)};
        if (pc < P_OUT) {  // (behind this wave's reads of the place it writes to)
            const int first = OP_Q + q_last(2 + pc - P_QS) + DIST;
            return {first < OP_GET_S + 1 ? OP_GET_S + 1 : first, OP_PUB_Q + 1};
        }
        if (pc < P_AS) return {DIST - 1, OP_Q + q_first(pc - P_OUT)};  // (the last MFMA of the previous chunk was its last op)
        if (pc < P_DEC) return {OP_GET_Q + 2, OP_P + (pc - P_AS)};
        if (pc < P_VS) return {OP_Q, lesser(OP_K + (pc - P_DEC), OP_BAR)};
        if (pc < P_VB) {
            const int t = pc - P_VS;
            return {OP_T + t_last(t) + DIST, OP_K + KT * (t / 2)};
        }
        if (pc < P_SB) {
            const int s = pc - P_VB;
            return {OP_T + t_last(2 * s + 1) + DIST, OP_P + 2 * s};
        }
        return {OP_K + KT + 2 * (pc - P_SB) + 1 + DIST, NOPS};
    }
    struct Table {
        int op[NPIECES];
        bool ok;
    };
    static constexpr Table make() {
        Table t{};
        bool done[NPIECES] = {};
        int left = NPIECES;
        t.ok = true;
        for (int op = 0; op < NOPS; op++) {
            const int quota = (left + (NOPS - op) - 1) / (NOPS - op);
            for (int n = 0;; n++) {
                int best = -1;
                for (int pc = 0; pc < NPIECES; pc++)
                    if (!done[pc] && window(pc).first <= op && (best < 0 || window(pc).end < window(best).end)) best = pc;
                if (best < 0) break;
                if (n >= quota && window(best).end > op + 1) break;
                if (window(best).end <= op) t.ok = false;  // window missed
                t.op[best] = op, done[best] = true, left--;
            }
        }
        if (left != 0) t.ok = false;
        // a slab of X is packed after the X of both its tiles (within an op the pieces run in index order)
        for (int s = 0; s < N_XB; s++)
            if (t.op[P_XB + s] < t.op[P_XC + 2 * s] || t.op[P_XB + s] < t.op[P_XC + 2 * s + 1]) t.ok = false;
        // what a piece takes out of this chunk's half of the stage is asked for before the barrier, in this chunk
        for (int i = 0; i < N_XC; i++)
            if (t.op[P_XC + i] - AHEAD < 0 || t.op[P_XC + i] - AHEAD >= OP_BAR) t.ok = false;
        for (int i = 0; i < N_VS; i++)
            if (t.op[P_VS + i] - AHEAD < 0 || t.op[P_VS + i] - AHEAD >= OP_BAR) t.ok = false;
        for (int i = 0; i < N_AS; i++)
            if (t.op[P_AS + i] >= NOPS) t.ok = false;
        for (int i = 0; i < N_DEC; i++)  // the barrier op replaces e^{gamma_C}
            if (t.op[P_DEC + i] >= OP_BAR) t.ok = false;
        return t;
    }
    static_assert(OP_PUB_S < OP_GET_S && OP_GET_S < OP_PUB_Q && OP_PUB_Q < OP_GET_Q && OP_GET_Q + 2 < OP_P && OP_K < OP_BAR, "order of the hand-overs");
};

struct KeysSchedule : KeysRules {
    static constexpr KeysRules::Table TABLE = KeysRules::make();
    static_assert(TABLE.ok, "no placement of the side work satisfies the windows");
    static constexpr int op_of(int pc) { return TABLE.op[pc]; }
};

__global__ __launch_bounds__(KEYS_WAVES* WAVE) void chunk_scan_keys_kernel(const ChunkParams p) {
    typedef KeysSchedule SCH;
    // the rows of q have a single buffer and the chunk a second workgroup barrier ("barrier Q", see the half-slice scan)
    constexpr int NL = KEYS_LOADERS;
    constexpr int KW = SCH::KW, KS = SCH::KS, KT = SCH::KT;
    // One half of the stage: [T diag(beta) 6 | P 6] | 64 rows of 32 columns of v | of k | 64 row scales of q | of
    // k for the state update | of k S0 | e^{gamma_C}
    constexpr int FRAGS = 12;
    constexpr int VROW = 64, VLD = VROW + 16;        // bytes per row of v, staged: the 32 columns that two workgroups share
    constexpr int V_UNITS = C * VROW / FRAG_BYTES;
    constexpr int QLD = 2 * K + 16;                  // bytes per staged row of q / k (16 bytes of padding against bank conflicts)
    constexpr int Q_UNITS = C * 2 * K / FRAG_BYTES;  // 1 KiB pieces of the rows of q; as many of k
    constexpr int V_OFF = FRAGS * FRAG_BYTES;
    constexpr int K_OFF = V_OFF + C * VLD;
    constexpr int QS_OFF = K_OFF + C * QLD;
    constexpr int KS_OFF = QS_OFF + C * 4;
    constexpr int CS_OFF = KS_OFF + C * 4;
    constexpr int EG_OFF = CS_OFF + C * 4;
    constexpr int STAGE_BYTES = EG_OFF + 16;
    constexpr int NF = FRAGS / NL, NV = V_UNITS / NL, NQ = Q_UNITS / NL, NLOAD = NF + NV + 2 * NQ;
    static_assert(FRAGS % NL == 0 && V_UNITS % NL == 0 && Q_UNITS % NL == 0, "the pieces must divide over the loader waves");
    // LDS: the stage halves | qstage | output staging [chunk parity][64 tokens][32 bytes] | hand-over [compute wave][4 tiles][64 lanes]; and its epochs
    constexpr int QSTAGE_OFF = 2 * STAGE_BYTES, OSTAGE_OFF = QSTAGE_OFF + C * QLD, XCH_OFF = OSTAGE_OFF + 2 * C * 32, XCH_WAVE = 4 * WAVE * 16;
    constexpr int LDS_BYTES = XCH_OFF + 2 * XCH_WAVE;
    static_assert(LDS_BYTES + 16 <= 160 * 1024 && STAGE_BYTES % 16 == 0, "stage exceeds LDS");
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_BYTES];
    __shared__ int epochs[2];
    uint8_t* const qstage = lds + QSTAGE_OFF;
    auto stage = [&](int c) { return lds + (c & 1) * STAGE_BYTES; };
    auto ostage_at = [&](int parity, int row) -> uint8_t* { return lds + OSTAGE_OFF + (parity * C + row) * 32; };

    const int lane = threadIdx.x % WAVE;
    const int wave = threadIdx.x / WAVE;

    // workgroup -> (sequence-head chain, column slice), as in the other scans: the slices of a chain on one XCD, the chains of a packed
    // batch dealt out longest first
    const int id = blockIdx.x;
    const int xcd = id % 8, rest = id / 8;
    const int vgroup = rest % p.scan_groups;  // 16 columns
    const int per_xcd = (p.N * p.H + 7) / 8;
    int n, h;
    {
        const int i = rest / p.scan_groups;
        if (p.cu_seqlens == nullptr) {
            const int chain = xcd * per_xcd + i;
            if (i >= per_xcd || chain >= p.N * p.H) return;  // whole workgroup
            n = chain / p.H, h = chain % p.H;
        } else {
            const int rank = 8 * i + ((xcd - i) % 8 + 8) % 8;
            if (i >= per_xcd || rank >= p.N * p.H) return;  // whole workgroup
            n = p.seq_order[rank / p.H], h = rank % p.H;
        }
    }
    int slot_begin, nchunks;
    int64_t b, seq_t0, seq_len;
    if (p.cu_seqlens == nullptr) {
        seq_len = p.pad_lens == nullptr ? p.T : min(max(p.pad_lens[n + 1] - p.pad_lens[n], 0), p.T);  // the last seq_len tokens of row n
        slot_begin = n * p.NT, nchunks = (int)((seq_len + C - 1) / C);
        b = n, seq_t0 = p.T - seq_len;
    } else {
        slot_begin = p.chunk_off[n], nchunks = p.chunk_off[n + 1] - slot_begin;
        int t0, len;
        packed_bounds(p.cu_seqlens, n, p.T, t0, len);
        b = 0, seq_t0 = t0, seq_len = min(len, nchunks * C);
    }
    const uint8_t* const rec = p.rec + ((int64_t)h * p.TC + slot_begin) * p.rec_bytes;

    // Zeros at the padding rows of a left-padded batch, for a caller that asks for them, while the first chunk is on its way, by the two
    // waves that have nothing else to do: the workgroups of a chain together in whole rows, 16 bytes a lane (see the other scans).
    auto zero_rows = [&](int w) {
        if (!p.zero_padding) return;
        const int per_row = p.V / 8, first = vgroup * 2 * WAVE + w * WAVE + lane;
        bf16x8 zero8;
#pragma unroll
        for (int e = 0; e < 8; e++) zero8[e] = (bf16_t)0.f;
        int row = first / per_row;
        bf16_t* at = p.o + b * p.o_stride_b + (int64_t)h * p.o_stride_h + 8 * (first % per_row) + (int64_t)row * p.o_stride_t;
#pragma unroll 4
        for (; row < (int)seq_t0; row += WAVE, at += WAVE * p.o_stride_t) *reinterpret_cast<bf16x8*>(at) = zero8;
    };
    if (wave == 5) {
        zero_rows(1);
        return;
    }
    if (wave == 4) {
        // ------------------------------ output store ------------------------------
        zero_rows(0);
        const int o_row = lane / 2, o_piece = lane % 2;  // 32 rows a store, 2 lanes a row
        bf16_t* const og = p.o + b * p.o_stride_b + (seq_t0 + o_row) * p.o_stride_t + (int64_t)h * p.o_stride_h + 16 * vgroup + 8 * o_piece;
        auto put_output = [&](int c) {
            const int valid = (int)min((int64_t)C, seq_len - (int64_t)c * C);
            bf16x8 x[2];
#pragma unroll
            for (int i = 0; i < 2; i++) x[i] = *reinterpret_cast<const bf16x8*>(ostage_at(c & 1, o_row + 32 * i) + 16 * o_piece);
#pragma unroll
            for (int i = 0; i < 2; i++)
                if (o_row + 32 * i < valid) *reinterpret_cast<bf16x8*>(og + ((int64_t)c * C + 32 * i) * p.o_stride_t) = x[i];
        };
        __syncthreads();
        for (int c = 0; c < nchunks; c++) {
            __syncthreads();  // barrier Q
            __syncthreads();  // the output of chunk c - 1 is staged
            if (c > 0) put_output(c - 1);
        }
        __syncthreads();
        if (nchunks > 0) put_output(nchunks - 1);
        return;
    }
    if (wave >= 2) {
        // ------------------------------ loader ------------------------------
        // The kind of every slot is known at compile time: a branch in these loops makes the compiler wait for every load in flight.
        // Addresses are a wave-uniform base of the chunk plus a 32-bit byte offset per lane.
        const int lw = __builtin_amdgcn_readfirstlane(wave < 4 ? wave - 2 : wave - 4);
        const int rot_f = vgroup % NF;  // the workgroups of a chain ask for different fragments at any one time
        auto frag_of = [&](int i) { return lw * NF + (i + rot_f < NF ? i + rot_f : i + rot_f - NF); };
        constexpr int Q_ROWS = C / Q_UNITS, Q_PIECES = WAVE / Q_ROWS;
        constexpr int V_ROWS = C / V_UNITS, V_PIECES = WAVE / V_ROWS;
        const int q_piece = lane % Q_PIECES, v_piece = lane % V_PIECES;
        const int hqk = qk_head_of(h, p.qk_div);
        const bf16_t* const qg = p.q + b * p.q_stride_b + seq_t0 * p.q_stride_t + (int64_t)hqk * p.q_stride_h;
        const bf16_t* const kg = p.k + b * p.k_stride_b + seq_t0 * p.k_stride_t + (int64_t)hqk * p.k_stride_h;
        const bf16_t* const vg = p.v + b * p.v_stride_b + seq_t0 * p.v_stride_t + (int64_t)h * p.v_stride_h + 32 * (vgroup / 2);
        bf16x8 buf0[NLOAD], buf1[NLOAD];
        struct Scalars {  // every loader wave carries the scales (identical values, identical LDS writes)
            float qs, ks, cs, eg;
        };
        Scalars sc0 = {0.f, 0.f, 0.f, 0.f}, sc1 = {0.f, 0.f, 0.f, 0.f};
        // slots: NF fragments | NV pieces of v | NQ of rows of k | NQ of rows of q
        auto src_of = [&](int c, int i) -> const uint8_t* {
            if (i < NF) return rec + (int64_t)c * p.rec_bytes + frag_of(i) * FRAG_BYTES + lane * 16;
            const int last = (int)min((int64_t)C, seq_len - (int64_t)c * C) - 1;  // a row past the end of the sequence is read from its last token
            int row0 = lane;
            asm volatile("" : "+v"(row0));  // (or the offsets of all slots are formed ahead of the loop and held in registers)
            if (i < NF + NV) {
                const uint32_t off = (uint32_t)min((lw * NV + i - NF) * V_ROWS + row0 / V_PIECES, last) * ((uint32_t)p.v_stride_t * 2u) + (uint32_t)v_piece * 16u;
                return reinterpret_cast<const uint8_t*>(vg + (int64_t)c * C * p.v_stride_t) + off;
            }
            const bool is_k = i < NF + NV + NQ;
            const int unit = lw * NQ + (i - NF - NV) % NQ;
            const uint32_t stride = (uint32_t)(is_k ? p.k_stride_t : p.q_stride_t) * 2u;
            const uint32_t off = (uint32_t)min(unit * Q_ROWS + row0 / Q_PIECES, last) * stride + (uint32_t)q_piece * 16u;
            return reinterpret_cast<const uint8_t*>((is_k ? kg : qg) + (int64_t)c * C * (is_k ? p.k_stride_t : p.q_stride_t)) + off;
        };
        auto dst_of = [&](uint8_t* st, int i) -> uint8_t* {
            if (i < NF) return st + frag_of(i) * FRAG_BYTES + lane * 16;
            if (i < NF + NV) return st + V_OFF + ((lw * NV + i - NF) * V_ROWS + lane / V_PIECES) * VLD + v_piece * 16;
            const int unit = lw * NQ + (i - NF - NV) % NQ;
            const int at = (lane / Q_PIECES) * QLD + q_piece * 16 + unit * Q_ROWS * QLD;
            if (i < NF + NV + NQ) return st + K_OFF + at;
            return qstage + at;
        };
        auto load_scalars = [&](Scalars& sc, int c) {
            const uint8_t* r = rec + (int64_t)c * p.rec_bytes;
            sc.qs = reinterpret_cast<const float*>(r + p.off_qs)[lane];
            sc.ks = reinterpret_cast<const float*>(r + p.off_ks)[lane];
            sc.cs = reinterpret_cast<const float*>(r + p.off_cs)[lane];
            sc.eg = *reinterpret_cast<const float*>(r + p.off_eg);
        };
        auto fetch = [&](int c, int i) -> bf16x8 { return *reinterpret_cast<const bf16x8*>(src_of(c, i)); };
        auto load = [&](bf16x8(&buf)[NLOAD], Scalars& sc, int c) {
#pragma unroll
            for (int i = 0; i < NLOAD; i++) buf[i] = fetch(c, i);
            load_scalars(sc, c);
        };
        // write chunk c to LDS and refill each register with chunk c2 right behind its write (the rows of q go last, behind barrier Q)
        auto store_and_reload = [&](bf16x8(&buf)[NLOAD], Scalars& sc, int c, int c2, auto reload_tag, auto barrier_q_tag) {
            constexpr bool reload = decltype(reload_tag)::value;
            constexpr bool barrier_q = decltype(barrier_q_tag)::value;
            uint8_t* const dst = stage(c);
            reinterpret_cast<float*>(dst + QS_OFF)[lane] = sc.qs;
            reinterpret_cast<float*>(dst + KS_OFF)[lane] = sc.ks;
            reinterpret_cast<float*>(dst + CS_OFF)[lane] = sc.cs;
            if (lane == 0) *reinterpret_cast<float*>(dst + EG_OFF) = sc.eg;
#pragma unroll
            for (int i = 0; i < NLOAD; i++) {
                if constexpr (barrier_q) {
                    if (i == NLOAD - NQ) __syncthreads();  // barrier Q: the compute waves have read the rows of q in the buffer
                }
                *reinterpret_cast<bf16x8*>(dst_of(dst, i)) = buf[i];
                if constexpr (reload) buf[i] = fetch(c2, i);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (reload) load_scalars(sc, c2);
        };
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        // chunks 0 (-> LDS now), 1 and 2 (in flight); even chunks use buf0, odd ones buf1
        if (nchunks > 0) {
            load(buf0, sc0, 0);
            if (nchunks > 1) load(buf1, sc1, 1);
            if (nchunks > 2) store_and_reload(buf0, sc0, 0, 2, yes, no);
            else store_and_reload(buf0, sc0, 0, 0, no, no);
        }
        __syncthreads();  // stage 0 holds chunk 0
        // Barrier of chunk c: the compute waves are done with its half and chunk c + 1 is in the other one.  Before it: write chunk c + 1
        // (its half was released by the barrier of chunk c - 1) and refill the freed registers with chunk c + 3.
        int c = 0;
        for (; c + 4 < nchunks; c += 2) {  // steady state: straight-line code, both reloads exist
            store_and_reload(buf1, sc1, c + 1, c + 3, yes, yes);
            __syncthreads();
            store_and_reload(buf0, sc0, c + 2, c + 4, yes, yes);
            __syncthreads();
        }
        for (; c < nchunks; c += 2) {  // the last (at most four) chunks; each has its barrier Q
            if (c + 1 < nchunks) {
                if (c + 3 < nchunks) store_and_reload(buf1, sc1, c + 1, c + 3, yes, yes);
                else store_and_reload(buf1, sc1, c + 1, 0, no, yes);
            } else {
                __syncthreads();
            }
            __syncthreads();
            if (c + 1 < nchunks) {
                if (c + 2 < nchunks) store_and_reload(buf0, sc0, c + 2, 0, no, yes);
                else __syncthreads();
                __syncthreads();
            }
        }
        __syncthreads();  // the last output tile
        return;
    }

    // ------------------------------ compute ------------------------------
    // Lane (j, g) = (lane % 16, lane / 16); operands A[j][8 g + 0..7], B[8 g + 0..7][j], accumulator D[4 g + r][j] of the 16x16x32 MFMA.
    // State tile t, register r: key KW kh + 32 (t / 2) + 8 g + 4 (t % 2) + r of column c0 + j; token tile t, register r: token 16 t + 4 g +
    // r; output tile, register r: column c0 + 4 g + r of token j of the tile.
    constexpr int NOPS = SCH::NOPS, OP_Q = SCH::OP_Q, OP_T = SCH::OP_T, OP_K = SCH::OP_K, OP_P = SCH::OP_P, OP_BAR = SCH::OP_BAR;
    constexpr int LA = SCH::LA;
    const int j16 = lane % 16, g = lane / 16;
    const int kh = __builtin_amdgcn_readfirstlane(wave);
    const int c0 = 16 * vgroup;
    f32x4* const own = reinterpret_cast<f32x4*>(lds + XCH_OFF + wave * XCH_WAVE) + lane;          // tile t at own[64 t]
    f32x4* const other = reinterpret_cast<f32x4*>(lds + XCH_OFF + (wave ^ 1) * XCH_WAVE) + lane;
    lds_flag_t* const own_flag = (lds_flag_t*)&epochs[wave];
    lds_flag_t* const other_flag = (lds_flag_t*)&epochs[wave ^ 1];
    pair_publish(own_flag, 0);

    f32x4 S[KT];
    auto st_key = [&](int t, int r) { return KW * kh + 32 * (t / 2) + 8 * g + 4 * (t % 2) + r; };
    const int64_t st_off = ((int64_t)n * p.H + h) * K * p.V + c0 + j16;
#pragma unroll
    for (int t = 0; t < KT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) S[t][r] = p.h0 != nullptr ? p.h0[st_off + (int64_t)st_key(t, r) * p.V] : 0.f;

    // logical output tile -> token tile: this wave finishes the tokens 32 kh .. 32 kh + 31
    auto token_tile = [&](int l) { return l < 2 ? 2 * kh + l : 2 * (1 - kh) + (l - 2); };
    auto lds_frag = [&](const uint8_t* st, auto opc) -> bf16x8 {
        constexpr int op = decltype(opc)::value;
        if constexpr (op < OP_Q) {  // rows of k
            constexpr int sl = SCH::s_slab(op), t = SCH::s_tile(op);
            return *reinterpret_cast<const bf16x8*>(st + K_OFF + (16 * t + j16) * QLD + (KW * kh + 32 * sl + 8 * g) * 2);
        } else if constexpr (op < OP_T) {  // rows of q
            constexpr int sl = SCH::s_slab(op - OP_Q), l = SCH::q_tile(op - OP_Q);
            return *reinterpret_cast<const bf16x8*>(qstage + (16 * token_tile(l) + j16) * QLD + (KW * kh + 32 * sl + 8 * g) * 2);
        } else if constexpr (op < OP_K) {  // T diag(beta)
            return reinterpret_cast<const bf16x8*>(st)[SCH::t_frag(op - OP_T) * WAVE + lane];
        } else if constexpr (op < OP_P) {
            // k^T: row j of key tile t is key 32 (t / 2) + 8 (j / 4) + 4 (t % 2) + j % 4 of the wave's; tokens 32 s + 4 g + 0..3 and + 16
            constexpr int sl = (op - OP_K) / KT, t = (op - OP_K) % KT;
            const bf16_t* km = reinterpret_cast<const bf16_t*>(st + K_OFF) + (32 * sl + 4 * g + j16 / 4) * (QLD / 2) + KW * kh + 32 * (t / 2) + 4 * (t % 2) + 8 * (j16 % 4);
            const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)km);
            const s16x4 c = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(km + 16 * (QLD / 2)));
            const bf16x4 a4 = __builtin_bit_cast(bf16x4, a), c4 = __builtin_bit_cast(bf16x4, c);
            bf16x8 r;
#pragma unroll
            for (int e = 0; e < 4; e++) r[e] = a4[e], r[4 + e] = c4[e];
            return r;
        } else {
            // P of tile l, slab s: fragments (0,0) (1,0) | (2,0) (2,1) (3,0) (3,1) of the record; the first tokens have no second slab and
            // take any fragment for it, their product with it is dropped
            constexpr int l = (op - OP_P) % 2, s = (op - OP_P) / 2;
            const int f = 6 + (l == 0 ? (s == 0 ? 2 : 3) * kh : 1 + (s == 0 ? 3 : 4) * kh);
            return reinterpret_cast<const bf16x8*>(st)[f * WAVE + lane];
        }
    };
    auto lds_eg = [&](const uint8_t* st) -> float { return *reinterpret_cast<const float*>(st + EG_OFF); };
    auto pack4x2 = [](const f32x4& a, const f32x4& c) {
        bf16x8 r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = (bf16_t)a[e], r[4 + e] = (bf16_t)c[e];
        return r;
    };
    auto out_tile = [&](const f32x4& acc, int parity, int l) {  // 4 columns of token j of the tile to the output staging
        bf16x4 o4;
#pragma unroll
        for (int e = 0; e < 4; e++) o4[e] = (bf16_t)acc[e];
        *reinterpret_cast<bf16x4*>(ostage_at(parity, 16 * token_tile(l) + j16) + 8 * g) = o4;
    };

    f32x4 accv[4], vt[4], acco[4];           // K S0 and then X, V~ by token tile; output by logical tile
    f32x4 sx[4], qx[2];                      // the other wave's halves
    bf16x8 sb[KS], xb[2], vb[2], vbs[2], fnext[LA];
    f32x4 ksr[4], csr[4];
    bf16x4 xvr[4];
    float egc, qsc[2] = {0.f, 0.f};
#pragma unroll
    for (int l = 0; l < 2; l++)
#pragma unroll
        for (int r = 0; r < 4; r++) acco[l][r] = 0.f;

    __syncthreads();  // stage 0 holds chunk 0
    egc = lds_eg(stage(0));
    static_for<0, LA>([&](auto i) { fnext[decltype(i)::value] = lds_frag(stage(0), i); });
#pragma unroll
    for (int s = 0; s < KS; s++) sb[s] = pack4x2(S[2 * s], S[2 * s + 1]);

    for (int c = 0; c < nchunks; c++) {
        const uint8_t* const st = stage(c);
        const uint8_t* const stn = stage(c + 1);
        bf16x8 fr[NOPS];
#pragma unroll
        for (int i = 0; i < LA; i++) fr[i] = fnext[i];
        __builtin_amdgcn_sched_barrier(0);

        auto run_piece = [&](auto pcc) {
            constexpr int pc = decltype(pcc)::value;
            if constexpr (pc < SCH::P_XC) {
                constexpr int t = pc - SCH::P_SS;
                own[WAVE * t] = accv[t];
            } else if constexpr (pc < SCH::P_XB) {  // X = V - diag(cs) K S0 (one sum of the halves in both waves: the same bits)
                constexpr int t = pc - SCH::P_XC;
#pragma unroll
                for (int e = 0; e < 4; e++) accv[t][e] = (float)xvr[t][e] - csr[t][e] * (accv[t][e] + sx[t][e]);
            } else if constexpr (pc < SCH::P_QS) {
                constexpr int s = pc - SCH::P_XB;
                xb[s] = pack4x2(accv[2 * s], accv[2 * s + 1]);
            } else if constexpr (pc < SCH::P_OUT) {
                constexpr int i = pc - SCH::P_QS;  // (into the other wave's place, which this one has read: its own waits for the next chunk)
                other[WAVE * i] = acco[2 + i];
            } else if constexpr (pc < SCH::P_AS) {
                constexpr int l = pc - SCH::P_OUT;
                if (c > 0) out_tile(acco[l], (c - 1) & 1, l);
            } else if constexpr (pc < SCH::P_DEC) {
                constexpr int l = pc - SCH::P_AS;
#pragma unroll
                for (int e = 0; e < 4; e++) acco[l][e] = (acco[l][e] + qx[l][e]) * qsc[l];
            } else if constexpr (pc < SCH::P_VS) {
                constexpr int t = pc - SCH::P_DEC;
#pragma unroll
                for (int e = 0; e < 4; e++) S[t][e] *= egc;
            } else if constexpr (pc < SCH::P_VB) {
                constexpr int t = pc - SCH::P_VS;
#pragma unroll
                for (int e = 0; e < 4; e++) vbs[t / 2][4 * (t % 2) + e] = (bf16_t)(vt[t][e] * ksr[t][e]);
            } else if constexpr (pc < SCH::P_SB) {
                constexpr int s = pc - SCH::P_VB;
                vb[s] = pack4x2(vt[2 * s], vt[2 * s + 1]);
            } else {
                constexpr int s = pc - SCH::P_SB;
                sb[s] = pack4x2(S[2 * s], S[2 * s + 1]);
                pin_regs(sb[s]);
            }
        };

        static_for<0, NOPS>([&](auto opc) {
            constexpr int op = decltype(opc)::value;
            if constexpr (op + LA < NOPS) fr[op + LA] = lds_frag(st, std::integral_constant<int, (op + LA < NOPS ? op + LA : 0)>{});
            if constexpr (op == OP_BAR) {
                __syncthreads();  // this wave is done with chunk c's half; chunk c + 1 is in the other one
                egc = lds_eg(stn);
            }
            if constexpr (op == OP_T) {
                // Barrier Q.  The MFMA before this point took the last fragment of q, and LDS reads return in order: no read of the q
                // buffer is outstanding, so the barrier needs no wait for the reads still in flight.
                static_assert(OP_T < OP_BAR && OP_Q >= LA, "barrier Q comes first and the prefetch across the chunk barrier holds no q");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (op >= OP_BAR) fnext[op >= OP_BAR ? op - OP_BAR : 0] = lds_frag(stn, std::integral_constant<int, (op >= OP_BAR ? op - OP_BAR : 0)>{});
            static_for<0, SCH::N_VS>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (SCH::op_of(SCH::P_VS + i) - SCH::AHEAD == op) ksr[i] = *reinterpret_cast<const f32x4*>(st + KS_OFF + (16 * i + 4 * g) * 4);
            });
            static_for<0, SCH::N_XC>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                if constexpr (SCH::op_of(SCH::P_XC + i) - SCH::AHEAD == op) {
                    csr[i] = *reinterpret_cast<const f32x4*>(st + CS_OFF + (16 * i + 4 * g) * 4);
                    xvr[i] = lds_read_tr4x16<false>(reinterpret_cast<const bf16_t*>(st + V_OFF), VLD / 2, 16 * i + 4 * g, 16 * (vgroup % 2), j16);
                }
            });
            if constexpr (op == SCH::OP_PUB_Q) {
#pragma unroll
                for (int l = 0; l < 2; l++) qsc[l] = reinterpret_cast<const float*>(st + QS_OFF)[16 * token_tile(l) + j16];
            }
            if constexpr (op == SCH::OP_GET_S) {
                pair_wait(other_flag, 2 * c + 1);
#pragma unroll
                for (int t = 0; t < 4; t++) sx[t] = other[WAVE * t];
            }
            if constexpr (op == SCH::OP_GET_Q) {
                pair_wait(other_flag, 2 * c + 2);
#pragma unroll
                for (int l = 0; l < 2; l++) qx[l] = own[WAVE * l];
            }
            static_for<0, SCH::NPIECES>([&](auto pcc) {
                if constexpr (SCH::op_of(decltype(pcc)::value) == op) run_piece(pcc);
            });
            if constexpr (op == SCH::OP_PUB_S) pair_publish(own_flag, 2 * c + 1);
            if constexpr (op == SCH::OP_PUB_Q) pair_publish(own_flag, 2 * c + 2);

            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            if constexpr (op < OP_Q) {  // K S0
                constexpr int sl = SCH::s_slab(op), t = SCH::s_tile(op);
                accv[t] = mfma_bf16(fr[op], sb[sl], sl == 0 ? zero : accv[t]);
            } else if constexpr (op < OP_T) {  // O^T = S0^T q^T
                constexpr int sl = SCH::s_slab(op - OP_Q), l = SCH::q_tile(op - OP_Q);
                acco[l] = mfma_bf16(sb[sl], fr[op], sl == 0 ? zero : acco[l]);
            } else if constexpr (op < OP_K) {  // V~ = T' X
                constexpr int t = SCH::t_tile(op - OP_T), sl = SCH::t_slab(op - OP_T);
                vt[t] = mfma_bf16(fr[op], xb[sl], sl == 0 ? zero : vt[t]);
            } else if constexpr (op < OP_P) {  // S = e^{gamma_C} S + k^T (row-scaled V~)
                constexpr int sl = (op - OP_K) / KT, t = (op - OP_K) % KT;
                S[t] = mfma_bf16(fr[op], vbs[sl], S[t]);
            } else {  // O^T += V~^T P^T
                constexpr int l = (op - OP_P) % 2, sl = (op - OP_P) / 2;
                const f32x4 sum = mfma_bf16(vb[sl], fr[op], acco[l]);
#pragma unroll
                for (int e = 0; e < 4; e++) acco[l][e] = sl == 0 || kh != 0 ? sum[e] : acco[l][e];
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    if (nchunks > 0) {
#pragma unroll
        for (int l = 0; l < 2; l++) out_tile(acco[l], (nchunks - 1) & 1, l);
    }
    __syncthreads();  // the store wave writes the last output tile
    if (p.ht != nullptr) {
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) p.ht[st_off + (int64_t)st_key(t, r) * p.V] = S[t][r];
    }
}

}  // namespace

int launch_scan_keys(ChunkParams& p, hipStream_t stream) {
    p.scan_groups = p.V / 16;
    const unsigned chains8 = (unsigned)(((int64_t)p.N * p.H + 7) / 8 * 8);
    hipLaunchKernelGGL(chunk_scan_keys_kernel, dim3(chains8 * p.scan_groups), dim3(KEYS_WAVES * WAVE), 0, stream, p);
    return (int)hipGetLastError();
}

}  // namespace gdn
