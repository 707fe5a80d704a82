// The two sweeps of the backward pass over the chunks of a sequence, on records that the prepare step writes for them
// (chunk_prepare32_kernel<K, true>): what the chunk-local gradients (gdn_chunk_bwd.hip) need from the states.  Counterpart
// upstream: the state recomputation and its reverse in fla's backward of chunk_gated_delta_rule, reached from
// lm_engine/modeling_utils/sequence_mixer_blocks/gated_deltanet/module.py:197-209 under autograd.
//
// Per chunk, with T = (I + A)^-1, P, gamma as in the forward (gdn_chunk.hip) and S0, dS1 the state the chunk starts from and
// the gradient of the state it ends with:
//     forward    X = V - diag(cs) K S0          V~ = T diag(beta) X       S1  = e^{gamma_C} S0 + K^T diag(ks) V~
//     reverse    X = P^T dO + diag(ks) K dS1    Y  = T^T X                dS0 = e^{gamma_C} dS1 + Q^T diag(qs) dO - K^T diag(beta cs) Y
//         cs = e^{gamma} / |k|     ks = e^{gamma_C - gamma} / |k|     qs = e^{gamma} scale / |q|
// Saved per chunk as bf16: S0 and V~, dS1 and Y.
//
// The reverse sweep as a forward scan over a "mirror" problem (reversed rows, gdn_chunk_bwd_prepare) takes two chunk steps per chunk
// and a kernel in front that forms P^T dO and its records; as one step it has 60 instead of 76 MFMAs per chunk (K = 128), none that
// only pass through the pipeline, P^T dO is neither rounded nor stored, and the records come out of the forward's prepare step.
// Kernel times when the sweeps were launches of their own, 32 columns to a workgroup, that kernel + forward sweep + reverse sweep against
// prepare + the two sweeps here: 4 x 4096 tokens, 16 heads,
// K = V = 128: 148 + 106 + 160 | 53 + 95 + 122 us; 11 packed sequences of 32768 tokens together: 339 + 225 + 330 | 108 + 190 +
// 243 us; 8 x 4096 tokens, 2 heads, K = 256, V = 512: 82 + 136 + 205 | 50 + 133 + 163 us.
//
// The workgroup is that of the half-slice scan (gdn_chunk_scan32.h): one (sequence, head) chain and one slice of 32 columns of V;
// two compute waves with 16 columns of the state each in 16x16x32 accumulators, four loader waves that bring the next chunks
// global -> registers -> LDS, a store wave that takes what is saved out of LDS.  What bounds it: the instruction stream of a
// compute wave (K = 128: 38 and 60 MFMAs per chunk), two of the four SIMDs carry none, and every slice of a chain loads the chunk's
// records and rows of q and k again.  At K = 128, where the chains fill the chip, a workgroup therefore owns 64 columns (NC = 4):
// a compute wave on every SIMD, one loader beside each, and the loaders also take out what is saved.  A step is then longer (one
// sequence of 4000 tokens, 16 heads 1.9 us where 32 columns take 1.2), but both sweeps of 4 x 4096 tokens, 16 heads fit the chip side by
// side: 205 -> 170 us, 817 MB at 4.8 TB/s where a plain copy reaches 5.2; 11 packed sequences, 32768 tokens 402 -> 348.  K = 256 at 64 columns does not fit the LDS.

#include <type_traits>

#include "gdn_chunk32_common.h"
#include "gdn_chunk_sweep.h"
#include "gdn_launch.h"

namespace gdn {

namespace {

constexpr int SWEEP_WAVES = 8;  // 0 1 compute | 2 3 loaders | 4 store | 5 exits at once | 6 7 loaders (as in the half-slice scan); NC = 4: 0 - 3 compute | 4 - 7 loaders
constexpr int SWEEP_LOADERS = 4;

// Order of the MFMAs of one chunk in a compute wave ("ops"), and where its side work goes; placement is the earliest-deadline
// walk of Scan16Rules (gdn_chunk_scan32.h), at compile time.  Groups:
//     reverse only: U = P^T dO (6) | K S (4 K/32) | reverse only: S += Q^T dO' (part A) | T X (6) | part B | S += K^T Y' (2 K/16)
// Part A runs while X is formed and part B while Y is: neither depends on them.  The token tiles and slabs of the
// triangular products are numbered in the order in which they become known: forwards in a forward sweep, backwards in a
// reverse sweep (T^T is upper triangular), so "logical" tile t is tile 3 - t and slab s is slab 1 - s there.
template <int K, bool REV, int NC>
struct SweepRules {
    static constexpr int KS = K / 32, KT = K / 16;
    static constexpr bool QS = REV && (K > 128 || (K == 128 && NC == 4));  // rows of q in a single buffer, freed by a barrier behind part B (see the kernel)
    static constexpr bool ONE_STAGING = REV && K > 128;                     // and so are the staged saves
    static constexpr int NU = REV ? 6 : 0, NS = 4 * KS, NK = 2 * KT;
    static constexpr int NQA = !REV ? 0 : K > 128 ? 2 * KT - 8 : KT, NQB = REV ? 2 * KT - NQA : 0;
    static constexpr int OP_U = 0, OP_S = OP_U + NU, OP_QA = OP_S + NS, OP_T = OP_QA + NQA, OP_QB = OP_T + 6, OP_K = OP_QB + NQB, NOPS = OP_K + NK;
    static constexpr int LA = K == 64 ? 6 : 10;  // operand fragments are read this many ops ahead of their MFMA
    static constexpr int OP_BAR = NOPS - LA;     // the chunk's barrier: every read of its stage half has been issued
    static constexpr int AHEAD = 4, DIST = 3;    // scales are read AHEAD ops before their piece, results taken DIST ops after their MFMA

    static constexpr int phys_t(int t) { return REV ? 3 - t : t; }
    static constexpr int phys_s(int s) { return REV ? 1 - s : s; }
    // op j of K S -> logical token tile, key slab: tiles 0 and 1 alternate through all slabs, then tiles 2 and 3
    static constexpr int s_tile(int j) { return 2 * (j / (2 * KS)) + j % 2; }
    static constexpr int s_slab(int j) { return (j % (2 * KS)) / 2; }
    static constexpr int s_last(int t) { return (t / 2) * 2 * KS + 2 * (KS - 1) + t % 2; }
    // op j of a triangular product -> logical tile, logical slab; fragment number in the record
    static constexpr int t_tile(int j) { return j < 4 ? j : j - 2; }
    static constexpr int t_slab(int j) { return j < 4 ? 0 : 1; }
    static constexpr int t_frag(int j) { return j < 2 ? j : j == 2 ? 2 : j == 3 ? 4 : j == 4 ? 3 : 5; }
    static constexpr int t_last(int t) { return t < 2 ? t : t + 2; }
    static constexpr int s_first(int s) { return s == 0 ? 0 : 4; }
    // op of S += Q^T dO': number j = KT slab + tile
    static constexpr int q_op(int j) { return j < NQA ? OP_QA + j : OP_QB + (j - NQA); }
    static constexpr int q_index(int op) { return op < OP_T ? op - OP_QA : NQA + (op - OP_QB); }

    // pieces: X of a token tile | X of a slab as operand | decay of a state tile | dO of a token tile with its rows scaled |
    // V~ or Y of a token tile with its rows scaled | the same, unscaled, to the staging | a state slab to the staging |
    // new state slab as operand
    static constexpr int N_XC = 4, N_XB = 2, N_DEC = KT, N_DO = REV ? 4 : 0, N_VS = 4, N_VST = 4, N_SST = KS, N_SB = KS;
    static constexpr int P_XC = 0, P_XB = P_XC + N_XC, P_DEC = P_XB + N_XB, P_DO = P_DEC + N_DEC, P_VS = P_DO + N_DO, P_VST = P_VS + N_VS,
                         P_SST = P_VST + N_VST, P_SB = P_SST + N_SST, NPIECES = P_SB + N_SB;
    struct Window {
        int first, end;  // the piece runs before the MFMA of an op in [first, end)
    };
    static constexpr int lesser(int a, int b) { return a < b ? a : b; }
    // state tiles 2 s, 2 s + 1 are final (the first slab is packed in its own chunk at the latest: the next begins with it)
    static constexpr int repack_first(int s) {
        const int op = OP_K + KT + 2 * s + 1 + DIST;
        return s == 0 ? lesser(op, NOPS - 1) : op;
    }
    static constexpr Window window(int pc) {
        if (pc < P_XB) {
            const int t = pc - P_XC;
            return {OP_S + s_last(t) + DIST, OP_T + s_first(t / 2)};
        }
        if (pc < P_DEC) {
            const int s = pc - P_XB;
            return {OP_S + s_last(2 * s + 1) + DIST, OP_T + s_first(s)};
        }
        if (pc < P_DO) {  // (the state's bf16 copy for this chunk is made by then)
            const int t = pc - P_DEC;
            return {OP_S + 2 * (t / 2) + 1, lesser(REV ? q_op(t) : OP_K + t, OP_BAR)};
        }
        if (pc < P_VS) return {AHEAD, q_op(KT * ((pc - P_DO) / 2))};
        if (pc < P_VST) {
            const int t = pc - P_VS;
            return {OP_T + t_last(t) + DIST, OP_K + KT * (t / 2)};
        }
        if (pc < P_SST) {
            // reverse: ahead of this chunk's barrier, behind which the store wave takes it; forward: behind it (the store wave
            // takes it behind the next one), where a chunk of 38 MFMAs has the room
            const int t = pc - P_VST, first = OP_T + t_last(t) + DIST;
            if (REV) return {ONE_STAGING && first < OP_K ? OP_K : first, OP_BAR};
            return {first < OP_BAR + 1 ? OP_BAR + 1 : first, NOPS};
        }
        if (pc < P_SB) {
            const int s = pc - P_SST;
            return {ONE_STAGING ? OP_K : OP_S + 2 * s + 1, lesser(OP_BAR, repack_first(s))};
        }
        const int s = pc - P_SB;  // what no longer fits this chunk is packed at the start of the next (whose first chunk packs twice)
        if (repack_first(s) >= NOPS) return {lesser(repack_first(s) - NOPS, OP_S + 2 * s - 1), OP_S + 2 * s};
        return {repack_first(s), NOPS};
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
        // a state slab goes to the staging from its operand registers: after they are packed, before they are packed again
        for (int s = 0; s < KS; s++) {
            if (t.op[P_SST + s] >= repack_first(s)) t.ok = false;
            if (repack_first(s) >= NOPS && t.op[P_SST + s] <= t.op[P_SB + s]) t.ok = false;
        }
        // what a piece takes out of this chunk's half of the stage is asked for before the barrier, in this chunk
        for (int i = 0; i < N_XC; i++)
            if (t.op[P_XC + i] - AHEAD < 0 || t.op[P_XC + i] - AHEAD >= OP_BAR) t.ok = false;
        for (int i = 0; i < N_VS; i++)
            if (t.op[P_VS + i] - AHEAD < 0 || t.op[P_VS + i] - AHEAD >= OP_BAR) t.ok = false;
        for (int i = 0; i < N_DO; i++)
            if (t.op[P_DO + i] - AHEAD < 0 || t.op[P_DO + i] >= OP_BAR) t.ok = false;
        for (int i = 0; i < N_DEC; i++)  // the barrier op replaces e^{gamma_C}
            if (t.op[P_DEC + i] >= OP_BAR) t.ok = false;
        return t;
    }
};

template <int K, bool REV, int NC>
struct SweepSchedule : SweepRules<K, REV, NC> {
    static constexpr typename SweepRules<K, REV, NC>::Table TABLE = SweepRules<K, REV, NC>::make();
    static_assert(TABLE.ok, "no placement of the side work satisfies the windows");
    static constexpr int op_of(int pc) { return TABLE.op[pc]; }
};

// One workgroup of a sweep.
template <int K, bool REV, int NC>
struct Sweep {
    typedef SweepSchedule<K, REV, NC> SCH;
    static_assert(NC == 2 || NC == 4, "compute waves of a workgroup");
    static constexpr int NCOL = 16 * NC;  // columns of a workgroup
    // K = 256, and K = 128 with four compute waves, reverse: two stage halves with the rows of q and of k do not fit the LDS.  The
    // rows of q, which a chunk needs for one group of MFMAs only, then get a single buffer and a second workgroup barrier per chunk
    // ("barrier Q"), and at K = 256 so do the staged saves: they are written between that barrier and the chunk's own and taken
    // out between the latter and the next barrier Q.
    static constexpr bool QS = SCH::QS;
    static constexpr int NL = SWEEP_LOADERS;
    static constexpr int KS = SCH::KS, KT = SCH::KT;
    // One half of the stage: fragments T' (forward: 6) or T^T | P^T (reverse: 12) | this workgroup's columns of 64 rows of v or
    // dO | rows of q (reverse) | of k | four vectors of 64 scales: ks | cs | e^{gamma_C} | - (forward), qs | ks | beta cs | e^{gamma_C}
    static constexpr int FRAGS = REV ? 12 : 6;
    static constexpr int VROW = 2 * NCOL;                   // bytes of a row of v / dO
    static constexpr int VLD = NC == 2 ? VROW : VROW + 16;  // and per staged one: rows 128 bytes apart would start on two banks only
    static constexpr int V_UNITS = C * VROW / FRAG_BYTES;   // 1 KiB pieces
    static constexpr int QLD = 2 * K + 16;                  // bytes per staged row of q / k (16 bytes of padding against bank conflicts)
    static constexpr int Q_UNITS = C * 2 * K / FRAG_BYTES;  // 1 KiB pieces of the rows of k; as many of q
    static constexpr int V_OFF = FRAGS * FRAG_BYTES;
    static constexpr int Q_OFF = V_OFF + C * VLD;  // not part of the stage halves when QS
    static constexpr int K_OFF = (REV && !QS) ? Q_OFF + C * QLD : Q_OFF;
    static constexpr int SC_OFF = K_OFF + C * QLD;
    static constexpr int STAGE_BYTES = SC_OFF + 4 * C * 4;
    static constexpr int XS_OFF = SC_OFF + C * 4;  // scale of K S's rows: cs, ks
    static constexpr int YS_OFF = SC_OFF + (REV ? 2 : 0) * C * 4;  // scale of V~'s or Y's rows in the state update: ks, beta cs
    static constexpr int EG_OFF = SC_OFF + (REV ? 3 : 2) * C * 4;
    static constexpr int NF = (FRAGS + NL - 1) / NL;  // fragment slots per loader wave (forward: 8 slots for 6 fragments, two of them twice)
    static constexpr int NV = V_UNITS / NL;
    static constexpr int NKR = Q_UNITS / NL;          // slots of rows of k; as many of q
    static constexpr int NQR = REV ? NKR : 0;
    static constexpr int NLOAD = NF + NV + NKR + NQR;
    static_assert(V_UNITS % NL == 0 && Q_UNITS % NL == 0, "the pieces must divide over the loader waves");
    // the staged saves, transposed: [columns][K + 8 keys], [columns][64 + 8 tokens]; a compute-wave lane writes 8 consecutive
    // keys (its operand register as it is) or 4 consecutive tokens of one column, the store wave turns them back into rows
    static constexpr int SCOL = (K + 8) * 2, VCOL = (C + 8) * 2, SBUFS = SCH::ONE_STAGING ? 1 : 2;
    // LDS: the stage halves | qstage | sstage | vstage
    static constexpr int QSTAGE_OFF = 2 * STAGE_BYTES, SSTAGE_OFF = QSTAGE_OFF + (QS ? C * QLD : 0), VSTAGE_OFF = SSTAGE_OFF + SBUFS * NCOL * SCOL;
    static constexpr int LDS_BYTES = VSTAGE_OFF + SBUFS * NCOL * VCOL;
    static_assert(LDS_BYTES <= 160 * 1024 && STAGE_BYTES % 16 == 0, "stage exceeds LDS");

    static __device__ __forceinline__ void run(const SweepParams& p, int id, uint8_t* lds);
};

template <int K, bool REV, int NC>
__device__ __forceinline__ void Sweep<K, REV, NC>::run(const SweepParams& p, int id, uint8_t* const lds) {
    uint8_t* const qstage = lds + QSTAGE_OFF;
    auto stage = [&](int i) { return lds + (i & 1) * STAGE_BYTES; };
    auto sstage = [&](int i) { return lds + SSTAGE_OFF + (SBUFS == 1 ? 0 : i & 1) * NCOL * SCOL; };
    auto vstage = [&](int i) { return lds + VSTAGE_OFF + (SBUFS == 1 ? 0 : i & 1) * NCOL * VCOL; };
    const int lane = threadIdx.x % WAVE;
    const int wave = threadIdx.x / WAVE;

    // workgroup -> (sequence-head chain, column slice), as in the scan of the forward: the slices of a chain on one XCD, the
    // chains of a packed batch dealt out longest first
    const int xcd = id % 8, rest = id / 8;
    const int groups = p.V / NCOL;
    const int vgroup = rest % groups;
    const int per_xcd = (p.N * p.H + 7) / 8;
    int n, h;
    {
        const int i = rest / groups;
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
    const int chain = n * p.H + h;
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
    nchunks = min(nchunks, p.save_nc);  // (the saves are laid out for save_nc chunks per chain: a longer prefix than the caller said writes none outside)
    const uint8_t* const rec = p.rec + ((int64_t)h * p.TC + slot_begin) * p.rec_bytes + (REV ? SWEEP_REC_REV : SWEEP_REC_FWD);
    const int64_t rec_scales = REV ? SWEEP_REC_REV_SCALES - SWEEP_REC_REV : SWEEP_REC_FWD_SCALES - SWEEP_REC_FWD;
    // the chunk that step i of the sweep works on
    auto chunk_of = [&](int i) { return REV ? nchunks - 1 - i : i; };

    // The staged saves on their way out: rows of 32 columns (64 bytes) of one contiguous block per chunk and slice, [slice][rows][32].
    // Lane group lane / 16 takes 8 columns of 16 consecutive rows through two transposing loads, 4 lanes per row; non-temporal, or
    // the saves push the rows that the loaders share out of the L2.  Y goes out with its rows in reverse order, as
    // gdn_chunk_bwd_local reads it.  Rows r0 .. r0 + 16 * COUNT - 1 of ROWS:
    auto flush = [&](const uint8_t* staged, int ld, bf16_t* dst, int r0, auto countc, auto rowsc, auto reversec) {
        constexpr int COUNT = decltype(countc)::value, ROWS = decltype(rowsc)::value;
        constexpr bool REVERSE = decltype(reversec)::value;
        const int l16 = lane % 16, piece = lane / 16;
        const bf16_t* const m = reinterpret_cast<const bf16_t*>(staged);
        bf16x8 x[COUNT];
#pragma unroll
        for (int i = 0; i < COUNT; i++) {
            const bf16x4 lo = lds_read_tr4x16<false>(m, ld, 8 * piece, r0 + 16 * i, l16);
            const bf16x4 hi = lds_read_tr4x16<false>(m, ld, 8 * piece + 4, r0 + 16 * i, l16);
#pragma unroll
            for (int e = 0; e < 4; e++) x[i][e] = lo[e], x[i][4 + e] = hi[e];
        }
#pragma unroll
        for (int i = 0; i < COUNT; i++) {
            const int row = r0 + 16 * i + l16;
            __builtin_nontemporal_store(x[i], reinterpret_cast<bf16x8*>(dst + (REVERSE ? ROWS - 1 - row : row) * 32 + 8 * piece));
        }
    };
    // slice `sl` of the workgroup's NC / 2
    auto state_at = [&](int i, int sl) { return p.save_state + ((int64_t)chain * p.save_nc + chunk_of(i)) * K * p.V + K * 32 * (vgroup * (NC / 2) + sl); };
    auto v_at_of = [&](int i, int sl) { return p.save_v + ((int64_t)chain * p.save_nc + chunk_of(i)) * C * p.V + C * 32 * (vgroup * (NC / 2) + sl); };
    constexpr std::integral_constant<int, K> k_rows{};
    constexpr std::integral_constant<int, C> c_rows{};
    constexpr std::integral_constant<bool, REV> v_reversed{};
    const bool is_store = NC == 2 && wave == 4;
    const bool is_loader = NC == 2 ? (wave == 2 || wave == 3 || wave >= 6) : wave >= 4;
    if (NC == 2 && wave == 5) return;
    if (is_store) {
        // ------------------------------ store ------------------------------
        constexpr std::integral_constant<int, 4> four{};
        auto flush_state = [&](int i) {
#pragma unroll 1
            for (int r = 0; r < K; r += 64) flush(sstage(i), SCOL / 2, state_at(i, 0), r, four, k_rows, std::false_type{});
        };
        auto flush_v = [&](int i) { flush(vstage(i), VCOL / 2, v_at_of(i, 0), 0, four, c_rows, v_reversed); };
        __syncthreads();
        for (int i = 0; i < nchunks; i++) {
            if constexpr (QS) __syncthreads();  // barrier Q: what was staged for step i - 1 has been taken out
            __syncthreads();                    // the state of step i is staged, and V~ of step i - 1 or Y of step i
            flush_state(i);
            if constexpr (REV) flush_v(i);
            else if (i > 0) flush_v(i - 1);
        }
        __syncthreads();
        if (!REV && nchunks > 0) flush_v(nchunks - 1);
        return;
    }
    if (is_loader) {
        // ------------------------------ loader ------------------------------
        // The kind of every slot is known at compile time: a branch in these loops makes the compiler wait for every load in
        // flight.  Addresses are a wave-uniform base of the chunk plus a 32-bit byte offset per lane.
        const int lw = __builtin_amdgcn_readfirstlane(NC == 2 && wave < 4 ? wave - 2 : wave - 4);
        // the slices of a chain ask for different lines at any one time (K = 256 has no registers for it)
        const int rot_f = vgroup % NF, rot_k = K > 128 ? 0 : vgroup % NKR;
        auto rotated = [](int i, int rot, int count) { return i + rot < count ? i + rot : i + rot - count; };
        auto frag_of = [&](int i) { return min(lw * NF + rotated(i, rot_f, NF), FRAGS - 1); };
        constexpr int Q_ROWS = C / Q_UNITS, Q_PIECES = WAVE / Q_ROWS;
        constexpr int V_ROWS = C / V_UNITS, V_PIECES = WAVE / V_ROWS;
        const int q_piece = lane % Q_PIECES, v_piece = lane % V_PIECES;
        const int hqk = qk_head_of(h, p.qk_div);
        const bf16_t* const qg = p.q + b * p.q_stride_b + seq_t0 * p.q_stride_t + (int64_t)hqk * p.q_stride_h;
        const bf16_t* const kg = p.k + b * p.k_stride_b + seq_t0 * p.k_stride_t + (int64_t)hqk * p.k_stride_h;
        const bf16_t* const vg = p.v + b * p.v_stride_b + seq_t0 * p.v_stride_t + (int64_t)h * p.v_stride_h + NCOL * vgroup;
        bf16x8 buf0[NLOAD], buf1[NLOAD];
        float sc0 = 0.f, sc1 = 0.f;  // this wave's scale vector, token `lane`
        // slots: NF fragments | NV pieces of v or dO | NKR of rows of k | NQR of rows of q
        auto src_of = [&](int c, int i) -> const uint8_t* {
            if (i < NF) return rec + (int64_t)c * p.rec_bytes + frag_of(i) * FRAG_BYTES + lane * 16;
            const int last = (int)min((int64_t)C, seq_len - (int64_t)c * C) - 1;  // a row past the end of the sequence is read from its last token
            int row0 = lane;
            asm volatile("" : "+v"(row0));  // (or the offsets of all slots are formed ahead of the loop and held in registers)
            if (i < NF + NV) {
                const uint32_t off = (uint32_t)min((lw * NV + i - NF) * V_ROWS + row0 / V_PIECES, last) * ((uint32_t)p.v_stride_t * 2u) + (uint32_t)v_piece * 16u;
                return reinterpret_cast<const uint8_t*>(vg + (int64_t)c * C * p.v_stride_t) + off;
            }
            const bool is_k = i < NF + NV + NKR;
            const int unit = lw * NKR + rotated((i - NF - NV) % NKR, rot_k, NKR);
            const uint32_t stride = (uint32_t)(is_k ? p.k_stride_t : p.q_stride_t) * 2u;
            const uint32_t off = (uint32_t)min(unit * Q_ROWS + row0 / Q_PIECES, last) * stride + (uint32_t)q_piece * 16u;
            return reinterpret_cast<const uint8_t*>((is_k ? kg : qg) + (int64_t)c * C * (is_k ? p.k_stride_t : p.q_stride_t)) + off;
        };
        auto dst_of = [&](uint8_t* st, int i) -> uint8_t* {
            if (i < NF) return st + frag_of(i) * FRAG_BYTES + lane * 16;
            if (i < NF + NV) return st + V_OFF + ((lw * NV + i - NF) * V_ROWS + lane / V_PIECES) * VLD + v_piece * 16;
            const int unit = lw * NKR + rotated((i - NF - NV) % NKR, rot_k, NKR);
            const int at = (lane / Q_PIECES) * QLD + q_piece * 16 + unit * Q_ROWS * QLD;
            if (i < NF + NV + NKR) return st + K_OFF + at;
            if constexpr (QS) return qstage + at;
            else return st + Q_OFF + at;
        };
        auto fetch = [&](int c, int i) -> bf16x8 { return *reinterpret_cast<const bf16x8*>(src_of(c, i)); };
        auto fetch_scale = [&](int c) -> float { return reinterpret_cast<const float*>(rec + (int64_t)c * p.rec_bytes + rec_scales)[lw * C + lane]; };
        auto load = [&](bf16x8(&buf)[NLOAD], float& sc, int i) {
            const int c = chunk_of(i);
#pragma unroll
            for (int s = 0; s < NLOAD; s++) buf[s] = fetch(c, s);
            sc = fetch_scale(c);
        };
        // write step i to LDS and refill each register for step i2 right behind its write (QS: the rows of q go last, behind barrier Q)
        auto store_and_reload = [&](bf16x8(&buf)[NLOAD], float& sc, int i, int i2, auto reload_tag, auto barrier_q_tag) {
            constexpr bool reload = decltype(reload_tag)::value;
            constexpr bool barrier_q = decltype(barrier_q_tag)::value;
            uint8_t* const dst = stage(i);
            const int c2 = chunk_of(i2);
            reinterpret_cast<float*>(dst + SC_OFF)[lw * C + lane] = sc;
#pragma unroll
            for (int s = 0; s < (QS ? NLOAD - NQR : NLOAD); s++) {
                *reinterpret_cast<bf16x8*>(dst_of(dst, s)) = buf[s];
                if constexpr (reload) buf[s] = fetch(c2, s);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (QS) {
                if constexpr (barrier_q) __syncthreads();  // barrier Q: the compute waves have read the rows of q in the buffer
#pragma unroll
                for (int s = NLOAD - NQR; s < NLOAD; s++) {
                    *reinterpret_cast<bf16x8*>(dst_of(dst, s)) = buf[s];
                    if constexpr (reload) buf[s] = fetch(c2, s);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if constexpr (reload) sc = fetch_scale(c2);
        };
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        // steps 0 (-> LDS now), 1 and 2 (in flight); even steps use buf0, odd ones buf1
        if (nchunks > 0) {
            load(buf0, sc0, 0);
            if (nchunks > 1) load(buf1, sc1, 1);
            if (nchunks > 2) store_and_reload(buf0, sc0, 0, 2, yes, no);
            else store_and_reload(buf0, sc0, 0, 0, no, no);
        }
        __syncthreads();  // stage[0] holds step 0
        // Four compute waves leave no SIMD for a store wave: the loaders take out what is staged, each half of the rows of one slice.
        auto flush_state = [&](int i) {
            if constexpr (NC == 4) flush(sstage(i) + 32 * (lw / 2) * SCOL, SCOL / 2, state_at(i, lw / 2), K / 2 * (lw % 2), std::integral_constant<int, K / 32>{}, k_rows, std::false_type{});
        };
        auto flush_v = [&](int i) {
            if constexpr (NC == 4) flush(vstage(i) + 32 * (lw / 2) * VCOL, VCOL / 2, v_at_of(i, lw / 2), C / 2 * (lw % 2), std::integral_constant<int, 2>{}, c_rows, v_reversed);
        };
        // what is complete behind the barrier of step i: the state of step i, Y of step i or V~ of step i - 1
        auto flush_step = [&](int i, auto v_tag) {
            flush_state(i);
            if constexpr (REV) flush_v(i);
            else if constexpr (decltype(v_tag)::value) flush_v(i - 1);
        };
        // Barrier of step i: the compute waves are done with stage[i & 1] and step i + 1 is in the other half.  Before it: write
        // step i + 1 (its half was released by the barrier of step i - 1) and refill the freed registers with step i + 3.
        int i = 0;
        if (NC == 4 && nchunks > 4) {  // two steps, the first of which has no V~ to take out yet
            store_and_reload(buf1, sc1, 1, 3, yes, yes);
            __syncthreads();
            flush_step(0, no);
            store_and_reload(buf0, sc0, 2, 4, yes, yes);
            __syncthreads();
            flush_step(1, yes);
            i = 2;
        }
        for (; i + 4 < nchunks; i += 2) {  // steady state: straight-line code, both reloads exist
            store_and_reload(buf1, sc1, i + 1, i + 3, yes, yes);
            __syncthreads();
            flush_step(i, yes);
            store_and_reload(buf0, sc0, i + 2, i + 4, yes, yes);
            __syncthreads();
            flush_step(i + 1, yes);
        }
        for (; i < nchunks; i += 2) {  // the last (at most four) steps; QS: each has its barrier Q
            if (i + 1 < nchunks) {
                if (i + 3 < nchunks) store_and_reload(buf1, sc1, i + 1, i + 3, yes, yes);
                else store_and_reload(buf1, sc1, i + 1, 0, no, yes);
            } else if constexpr (QS) {
                __syncthreads();
            }
            __syncthreads();
            if (i == 0) flush_step(i, no);
            else flush_step(i, yes);
            if (i + 1 < nchunks) {
                if (i + 2 < nchunks) store_and_reload(buf0, sc0, i + 2, 0, no, yes);
                else if constexpr (QS) __syncthreads();
                __syncthreads();
                flush_step(i + 1, yes);
            }
        }
        __syncthreads();  // the last staged V~
        if (!REV && nchunks > 0) flush_v(nchunks - 1);
        return;
    }

    // ------------------------------ compute ------------------------------
    // Lane (j, g) = (lane % 16, lane / 16); operands A[j][8 g + 0..7], B[8 g + 0..7][j], accumulator D[4 g + r][j] of the 16x16x32
    // MFMA.  State tile t, register r: key 32 (t / 2) + 8 g + 4 (t % 2) + r of column c0 + j; token tile t, register r: token
    // 16 t + 4 g + r.  (The orders in which operands enumerate their reduction index: gdn_chunk_scan32.h.)
    constexpr int NOPS = SCH::NOPS, OP_S = SCH::OP_S, OP_QA = SCH::OP_QA, OP_T = SCH::OP_T, OP_QB = SCH::OP_QB, OP_K = SCH::OP_K, OP_BAR = SCH::OP_BAR;
    constexpr int LA = SCH::LA;
    const int j16 = lane % 16, g = lane / 16;
    const int half = wave;  // 0 .. NC - 1
    const int c0 = NCOL * vgroup + 16 * half;
    f32x4 S[KT];
    const int64_t st_off = (int64_t)chain * K * p.V + c0 + j16;
    auto st_key = [&](int t, int r) { return 32 * (t / 2) + 8 * g + 4 * (t % 2) + r; };
#pragma unroll
    for (int t = 0; t < KT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) S[t][r] = p.s_in != nullptr ? p.s_in[st_off + (int64_t)st_key(t, r) * p.V] : 0.f;

    // 8 tokens of one key (of q or k) per lane: row j of key tile t is key 32 (t / 2) + 8 (j / 4) + 4 (t % 2) + j % 4
    auto rows_transposed = [&](const uint8_t* rows, int t, int s) -> bf16x8 {
        const bf16_t* m = reinterpret_cast<const bf16_t*>(rows) + (32 * s + 4 * g + j16 / 4) * (QLD / 2) + 32 * (t / 2) + 4 * (t % 2) + 8 * (j16 % 4);
        const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)m);
        const s16x4 c = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(m + 16 * (QLD / 2)));
        const bf16x4 a4 = __builtin_bit_cast(bf16x4, a), c4 = __builtin_bit_cast(bf16x4, c);
        bf16x8 r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = a4[e], r[4 + e] = c4[e];
        return r;
    };
    auto lds_frag = [&](const uint8_t* st, auto opc) -> bf16x8 {
        constexpr int op = decltype(opc)::value;
        if constexpr (op < OP_S) {  // P^T
            return reinterpret_cast<const bf16x8*>(st)[(6 + SCH::t_frag(op)) * WAVE + lane];
        } else if constexpr (op < OP_QA) {  // rows of k
            constexpr int jj = op - OP_S, sl = SCH::s_slab(jj), tt = SCH::phys_t(SCH::s_tile(jj));
            return *reinterpret_cast<const bf16x8*>(st + K_OFF + (16 * tt + j16) * QLD + (32 * sl + 8 * g) * 2);
        } else if constexpr (op >= OP_T && op < OP_QB) {  // T diag(beta) or T^T
            return reinterpret_cast<const bf16x8*>(st)[SCH::t_frag(op - OP_T) * WAVE + lane];
        } else if constexpr (op >= OP_K) {
            constexpr int jj = op - OP_K;
            return rows_transposed(st + K_OFF, jj % KT, SCH::phys_s(jj / KT));
        } else {
            constexpr int jj = SCH::q_index(op);
            return rows_transposed(QS ? qstage : st + Q_OFF, jj % KT, SCH::phys_s(jj / KT));
        }
    };
    auto rows_of_v = [&](const uint8_t* st, int tile) -> bf16x4 {  // tokens 16 tile + 4 g + 0..3 of this lane's column
        return lds_read_tr4x16<false>(reinterpret_cast<const bf16_t*>(st + V_OFF), VLD / 2, 16 * tile + 4 * g, 16 * half, j16);
    };
    auto lds_eg = [&](const uint8_t* st) -> float { return *reinterpret_cast<const float*>(st + EG_OFF); };
    auto pack4x2 = [](const f32x4& a, const f32x4& c) {
        bf16x8 r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = (bf16_t)a[e], r[4 + e] = (bf16_t)c[e];
        return r;
    };

    f32x4 accv[4], accu[REV ? 4 : 1], vt[4];     // by logical token tile: K S and then X, P^T dO, V~ or Y
    bf16x8 sb[KS], xb[2], vbs[2], fnext[LA];     // operands: state, X and scaled V~ / Y by logical slab
    bf16x8 dob[REV ? 2 : 1], dobn[REV ? 2 : 1], dos[REV ? 2 : 1];  // dO and scaled dO by logical slab
    f32x4 ysr[4], xsr[4], qsr[REV ? 4 : 1];      // row scales on their way to the pieces that use them
    bf16x4 xvr[4];                               // and rows of v
    float egc;
    auto load_do = [&](const uint8_t* st, int s) {  // dO of logical slab s as operand: tokens 32 s' + 4 g + 0..3 and + 16
        const bf16x4 lo = rows_of_v(st, 2 * SCH::phys_s(s)), hi = rows_of_v(st, 2 * SCH::phys_s(s) + 1);
        bf16x8 r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = lo[e], r[4 + e] = hi[e];
        return r;
    };

    __syncthreads();  // stage[0] holds step 0
    egc = lds_eg(stage(0));
    if constexpr (REV) dobn[0] = load_do(stage(0), 0), dobn[1] = load_do(stage(0), 1);
    static_for<0, LA>([&](auto i) { fnext[decltype(i)::value] = lds_frag(stage(0), i); });
#pragma unroll
    for (int s = 0; s < KS; s++) sb[s] = pack4x2(S[2 * s], S[2 * s + 1]);

    for (int i = 0; i < nchunks; i++) {
        const uint8_t* const st = stage(i);
        const uint8_t* const stn = stage(i + 1);
        uint8_t* const s_at = sstage(i) + (16 * half + j16) * SCOL + (8 * g) * 2;
        uint8_t* const v_at = vstage(i) + (16 * half + j16) * VCOL + (4 * g) * 2;
        bf16x8 fr[NOPS];
#pragma unroll
        for (int f = 0; f < LA; f++) fr[f] = fnext[f];
        if constexpr (REV) dob[0] = dobn[0], dob[1] = dobn[1];
        __builtin_amdgcn_sched_barrier(0);

        auto run_piece = [&](auto pcc) {
            constexpr int pc = decltype(pcc)::value;
            if constexpr (pc < SCH::P_XB) {
                constexpr int t = pc - SCH::P_XC;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if constexpr (REV) accv[t][e] = accu[t][e] + xsr[t][e] * accv[t][e];
                    else accv[t][e] = (float)xvr[t][e] - xsr[t][e] * accv[t][e];
                }
            } else if constexpr (pc < SCH::P_DEC) {
                // logical tiles 2 s, 2 s + 1 as the physical order of the slab: the tile with the lower tokens first
                constexpr int s = pc - SCH::P_XB;
                xb[s] = pack4x2(accv[REV ? 2 * s + 1 : 2 * s], accv[REV ? 2 * s : 2 * s + 1]);
            } else if constexpr (pc < SCH::P_DO) {
                constexpr int t = pc - SCH::P_DEC;
#pragma unroll
                for (int e = 0; e < 4; e++) S[t][e] *= egc;
            } else if constexpr (pc < SCH::P_VS) {
                constexpr int t = pc - SCH::P_DO, at = REV ? 1 - t % 2 : t % 2;  // half of the slab's operand that tile t is
#pragma unroll
                for (int e = 0; e < 4; e++) dos[t / 2][4 * at + e] = (bf16_t)((float)dob[t / 2][4 * at + e] * qsr[t][e]);
            } else if constexpr (pc < SCH::P_VST) {
                constexpr int t = pc - SCH::P_VS, at = REV ? 1 - t % 2 : t % 2;
#pragma unroll
                for (int e = 0; e < 4; e++) vbs[t / 2][4 * at + e] = (bf16_t)(vt[t][e] * ysr[t][e]);
            } else if constexpr (pc < SCH::P_SST) {
                constexpr int t = pc - SCH::P_VST;
                bf16x4 x;
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = (bf16_t)vt[t][e];
                *reinterpret_cast<bf16x4*>(v_at + (16 * SCH::phys_t(t)) * 2) = x;
            } else if constexpr (pc < SCH::P_SB) {
                constexpr int s = pc - SCH::P_SST;
                *reinterpret_cast<bf16x8*>(s_at + (32 * s) * 2) = sb[s];
            } else {
                constexpr int s = pc - SCH::P_SB;
                sb[s] = pack4x2(S[2 * s], S[2 * s + 1]);
                pin_regs(sb[s]);  // (or the compiler moves all of them behind the last MFMA)
            }
        };

        static_for<0, NOPS>([&](auto opc) {
            constexpr int op = decltype(opc)::value;
            if constexpr (op + LA < NOPS) fr[op + LA] = lds_frag(st, std::integral_constant<int, (op + LA < NOPS ? op + LA : 0)>{});
            if constexpr (op == OP_BAR) {
                __syncthreads();  // this wave is done with this step's half; the next step is in the other one
                egc = lds_eg(stn);
            }
            if constexpr (QS && op == OP_K) {
                // Barrier Q.  The MFMA before this point took the last fragment of q, and LDS reads return in order: no read of
                // the q buffer is outstanding, so the barrier needs no wait for the reads still in flight.
                static_assert(!QS || OP_K < OP_BAR, "barrier Q comes first");
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (op >= OP_BAR) {
                constexpr int nx = op >= OP_BAR ? op - OP_BAR : 0;
                fnext[nx] = lds_frag(stn, std::integral_constant<int, nx>{});
                if constexpr (REV && nx < 2) dobn[nx] = load_do(stn, nx);
            }
            static_for<0, SCH::N_VS>([&](auto ic) {
                constexpr int t = decltype(ic)::value;
                if constexpr (SCH::op_of(SCH::P_VS + t) - SCH::AHEAD == op)
                    ysr[t] = *reinterpret_cast<const f32x4*>(st + YS_OFF + (16 * SCH::phys_t(t) + 4 * g) * 4);
            });
            static_for<0, SCH::N_XC>([&](auto ic) {
                constexpr int t = decltype(ic)::value;
                if constexpr (SCH::op_of(SCH::P_XC + t) - SCH::AHEAD == op) {
                    xsr[t] = *reinterpret_cast<const f32x4*>(st + XS_OFF + (16 * SCH::phys_t(t) + 4 * g) * 4);
                    if constexpr (!REV) xvr[t] = rows_of_v(st, t);
                }
            });
            static_for<0, SCH::N_DO>([&](auto ic) {
                constexpr int t = decltype(ic)::value;
                if constexpr (SCH::op_of(SCH::P_DO + t) - SCH::AHEAD == op)
                    qsr[t] = *reinterpret_cast<const f32x4*>(st + SC_OFF + (16 * SCH::phys_t(t) + 4 * g) * 4);
            });
            static_for<0, SCH::NPIECES>([&](auto pcc) {
                if constexpr (SCH::op_of(decltype(pcc)::value) == op) run_piece(pcc);
            });

            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            if constexpr (op < OP_S) {  // U = P^T dO
                constexpr int t = SCH::t_tile(op), s = SCH::t_slab(op);
                accu[t] = mfma_bf16(fr[op], dob[s], s == 0 ? zero : accu[t]);
            } else if constexpr (op < OP_QA) {  // K S
                constexpr int jj = op - OP_S, sl = SCH::s_slab(jj), t = SCH::s_tile(jj);
                accv[t] = mfma_bf16(fr[op], sb[sl], sl == 0 ? zero : accv[t]);
            } else if constexpr (op >= OP_T && op < OP_QB) {  // V~ = T diag(beta) X, Y = T^T X
                constexpr int jj = op - OP_T, t = SCH::t_tile(jj), s = SCH::t_slab(jj);
                vt[t] = mfma_bf16(fr[op], xb[s], s == 0 ? zero : vt[t]);
            } else if constexpr (op >= OP_K) {  // S += K^T (scaled V~ or Y)
                constexpr int jj = op - OP_K;
                S[jj % KT] = mfma_bf16(fr[op], vbs[jj / KT], S[jj % KT]);
            } else {  // S += Q^T (scaled dO)
                constexpr int jj = SCH::q_index(op);
                S[jj % KT] = mfma_bf16(fr[op], dos[jj / KT], S[jj % KT]);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    __syncthreads();  // the store wave takes the last V~
    if (p.s_out != nullptr) {
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) p.s_out[st_off + (int64_t)st_key(t, r) * p.V] = S[t][r];
    }
}

// Both sweeps in one launch: neither needs anything of the other, so with fewer workgroups than compute units they run side by
// side, and with more the forward sweep's first workgroups start on the units that the reverse sweep's last ones leave idle.  The
// reverse sweep comes first, its chunks are the longer ones.  `first`: the number of the launch's first workgroup.  Kernel times at 32
// columns to a workgroup, two launches | one: 4 x 4096 tokens, 16 heads, K = V = 128 (256 workgroups a sweep) 220 | 208 us, 2 x 4096 142 | 107, 2184 tokens 77 | 45;
// 11 packed sequences, 32768 tokens 428 | 397; 9000 tokens, 3 heads, K = 256, V = 512 467 | 289.  Slower only where one launch takes
// forward workgroups their place, see launch_sweeps.  With many rounds of workgroups a sweep it is the gap between the launches that
// goes: at 2 x 2048 tokens, 32 heads, V = 256 (512) the kernels alone take 196 | 202 us, calls of gdn_chunk_bwd_sweeps back to back 203
// | 201; 8 x 2048, 16 heads, V = 128 265 | 256; 4 x 1024, 32 heads, V = 256 (1024) 187 | 186; 32 x 512, 16 heads (2048) 291 | 282.
template <int K, int NC>
__global__ __launch_bounds__(SWEEP_WAVES* WAVE) void chunk_sweeps_kernel(const SweepParams fwd, const SweepParams rev, unsigned groups, unsigned first) {
    constexpr int LDS = Sweep<K, true, NC>::LDS_BYTES > Sweep<K, false, NC>::LDS_BYTES ? Sweep<K, true, NC>::LDS_BYTES : Sweep<K, false, NC>::LDS_BYTES;
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS];
    const unsigned id = blockIdx.x + first;
    if (id < groups) Sweep<K, true, NC>::run(rev, id, lds);
    else Sweep<K, false, NC>::run(fwd, id - groups, lds);
}

template <int K, bool REV>
__global__ __launch_bounds__(SWEEP_WAVES* WAVE) void chunk_sweep_kernel(const SweepParams p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[Sweep<K, REV, 2>::LDS_BYTES];
    Sweep<K, REV, 2>::run(p, blockIdx.x, lds);
}

}  // namespace

// Columns of a workgroup at K = 128; `longest`: chunks of the longest sequence, `chunks`: of all rows together.
//
// 64 columns are half as many workgroups whose step is about 1.45 times as long.  That pays unless the longest chain is what the launch waits
// for: its chunks against the chunks that a CU is given at 32 columns (of one sweep).  Records and sweeps at 32 | 64 columns, by that ratio.
// Rows of one length: 2 x 2048 tokens, 16 heads (2.0) 63 | 82 us, 2048 tokens, 36 heads (1.8) 90 | 88, 3 x 2048, 16 heads (1.3) 96 | 89, 5 x
// 2048 (0.8) 135 | 125, 8 x 2048 (0.5) 252 | 198, 128 x 128 (0.06) 407 | 283.  Packed ones, dealt out longest first, which smaller workgroups
// fill up better: 3 sequences, 18000 tokens (2.1) 317 | 371, 6 of 11776 (1.4) 160 | 174, 10 of 13312 (1.2) 201 | 193, 3 of 2548, 32 heads, V
// = 256 (0.8) 128 | 107, 24 of 20000 (0.4) 338 | 261.  Tokens behind the last sequence are nobody's: the rows count for no more than
// the sequences can have (one of 4000 tokens in a row of 32768: 97 | 140).
//
// Left-padded rows, whose lengths the host does not have here: one of them may be all there is, and the rows' chains go to the XCDs in the
// order of the batch.  Where the chains of one row do not fit their XCD side by side at 32 columns, both sweeps of it, they queue for
// its CUs and 64 columns win however the tokens lie: 26 x 2048, 5 heads, V = 128, one row full, the others 64 tokens 92 | 85, every length 189
// | 169; 8 x 2048, 16 heads 168 | 135, V = 64 98 | 92; 43 x 2048, 3 heads, V = 256 109 | 96.  Where they fit, 32 columns are the
// safe side: 32 x 2048, 4 heads, V = 128 86 | 102 and 189 | 159; 16 x 2048, 8 heads, V = 64 80 | 102 and 117 | 125; 48 x 2048, 2 heads, V =
// 256 84 | 94 and 237 | 191.
int sweep_columns_k128(int N, int H, int V, int longest, int64_t chunks, bool packed, bool padded, int num_cus) {
    const int64_t slices = V / 32, possible = (int64_t)N * longest;
    if (V % 64 != 0) return 32;
    if (padded) {
        const int64_t per_xcd = ((int64_t)N * H + 7) / 8, chains = H < per_xcd ? H : per_xcd;  // of one row, on one XCD
        if (2 * chains * slices <= num_cus / 8) return 32;
    }
    if (chunks > possible) chunks = possible;
    return 4 * (int64_t)longest * num_cus < (packed || padded ? 5 : 7) * chunks * H * slices ? 64 : 32;
}

namespace {

template <int K, int NC>
int launch_both(const SweepParams& fwd, const SweepParams& rev, hipStream_t stream) {
    const int64_t chains8 = ((int64_t)fwd.N * fwd.H + 7) / 8 * 8;
    const unsigned groups = (unsigned)(chains8 * (fwd.V / (16 * NC)));
    const dim3 block(SWEEP_WAVES * WAVE);
    // (a launch holds at most 2^32 - 1 threads)
    const int launches = (uint64_t)2 * groups * block.x >> 32 ? 2 : 1;
    for (int i = 0; i < launches; i++) {
        hipLaunchKernelGGL((chunk_sweeps_kernel<K, NC>), dim3(2 / launches * groups), block, 0, stream, fwd, rev, groups, i * groups);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
    }
    return GDN_OK;
}

template <int K>
int launch_sweeps(const SweepParams& fwd, const SweepParams& rev, hipStream_t stream) {
    const int64_t chains8 = ((int64_t)fwd.N * fwd.H + 7) / 8 * 8;
    const unsigned groups = (unsigned)(chains8 * (fwd.V / 32));
    if constexpr (K == 64) {
        // Here two forward workgroups fit a compute unit (59 KB of LDS) and only one of both sweeps' (90 KB).  64 x 1024 tokens, 4
        // heads, two launches | one: 82 | 89 us; a packed batch, of uneven chains, gains all the same (30000 tokens, 16 heads 178 | 153).
        if (fwd.cu_seqlens == nullptr && groups > (unsigned)compute_units()) {
            const dim3 block(SWEEP_WAVES * WAVE);
            hipLaunchKernelGGL((chunk_sweep_kernel<K, false>), dim3(groups), block, 0, stream, fwd);
            if (hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
            hipLaunchKernelGGL((chunk_sweep_kernel<K, true>), dim3(groups), block, 0, stream, rev);
            return (int)hipGetLastError();
        }
    }
    if constexpr (K == 128) {
        const bool packed = fwd.cu_seqlens != nullptr;
        if (sweep_columns_k128(fwd.N, fwd.H, fwd.V, fwd.save_nc, packed ? fwd.T / C : (int64_t)fwd.N * fwd.NT, packed, fwd.pad_lens != nullptr, compute_units()) == 64)
            return launch_both<K, 4>(fwd, rev, stream);
    }
    return launch_both<K, 2>(fwd, rev, stream);
}

}  // namespace

int launch_chunk_sweeps(const SweepParams& fwd, const SweepParams& rev, int K, hipStream_t stream) {
    if (K == 64) return launch_sweeps<64>(fwd, rev, stream);
    if (K == 128) return launch_sweeps<128>(fwd, rev, stream);
    if (K == 256) return launch_sweeps<256>(fwd, rev, stream);
    return GDN_ERR_UNSUPPORTED;
}

}  // namespace gdn
