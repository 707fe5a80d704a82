// Types and device helpers shared by the chunked-forward kernels of the gated delta rule.
#pragma once

#include "gdn_common.h"

namespace gdn {

constexpr int C = 64;  // chunk length
constexpr int GDN_CYCLE_BUDGET_SLOTS = 64;  // sampled workgroups of the measurement build
constexpr int GDN_LOCAL_CYCLE_SLOTS = 32;   // of them the chunk-local backward kernel uses two each (16 counters per workgroup)
constexpr int PREP_THREADS = 256;
constexpr int FRAG_BYTES = WAVE * 16;  // one MFMA operand fragment: 8 bf16 per lane

// head of q and k that value head h reads
__host__ __device__ inline int qk_head_of(int h, int qk_div) { return qk_div > 1 ? h / qk_div : h; }

struct ChunkParams {
    const bf16_t* q;
    const bf16_t* k;
    const bf16_t* v;
    const void* beta;
    const float* g;
    const float* h0;
    float* ht;
    bf16_t* o;
    const int32_t* cu_seqlens;  // packed sequences (B == 1), else NULL
    const int32_t* pad_lens;    // left-padded batch: prefix sums of the valid lengths, else NULL
    int32_t* chunk_off;  // [N + 1] prefix of chunks per sequence (packed input only)
    int32_t* seq_order;  // [N] the sequences by decreasing number of chunks (packed input only)
    uint8_t* rec;        // workspace records, [H][TC]
    int64_t q_stride_b, q_stride_t, q_stride_h;
    int64_t k_stride_b, k_stride_t, k_stride_h;
    int64_t v_stride_b, v_stride_t, v_stride_h;
    int64_t o_stride_b, o_stride_t, o_stride_h;
    int B, T, H, V, N;
    int qk_div;  // value heads per head of q and k (grouped value attention): head h reads q and k of head h / qk_div
    // Mirror reads (gdn_chunk_saves.mirror_reads, the scan without output): the sequence the scan walks is
    // the caller's sequence backwards, every chunk twice - chunk 2 r takes its rows of k from k and of v from v, chunk
    // 2 r + 1 from k2 and v2, both as tokens 64 (NT / 2 - 1 - r) + 63 - row of those tensors ([N, T / 2, H, .]).
    int mirror;
    int save_sliced;  // bf16 staged saves: [entry][V / 32 slices][rows][32] instead of [entry][rows][V]
    const bf16_t* k2;
    const bf16_t* v2;
    int64_t k2_stride_b, k2_stride_t, k2_stride_h;
    int64_t v2_stride_b, v2_stride_t, v2_stride_h;
    int NT;  // chunks per sequence (fixed-length input)
    int TC;  // chunk slots per head
    int beta_dtype;
    int l2norm;
    float scale;
    uint32_t rec_bytes, off_qs, off_ks, off_cs, off_p, off_eg;
    int scan_groups;  // workgroups per (sequence, head) in the scan kernel
    // training support: when set, the scan also writes the fp32 state every
    // chunk starts from, [N * H][save_nc][K][V], and V~ of every chunk, [N * H][save_nc][64][V]
    float* save_state;
    float* save_vnew;
    int save_nc;
    int save_every;    // only chunks c with c % save_every == 0 are saved, as entry c / save_every ...
    int save_reverse;  // ... or, when set, as entry save_nc - 1 - c / save_every
    const int32_t* row_order;  // left-padded rows of given records: the order in which the rows' chains are dealt out (or NULL)
    int save_state_bf16, save_vnew_bf16;  // that array is bf16 (the pointer then points at bf16 data); staged saves only
    int no_output;     // the scan writes no output (gdn_chunk_saves.no_output); staged saves only
    int records_given;  // the records are already in place: prepare is not run
    int32_t* ready;     // [H][TC] one flag per record, for the launch that runs prepare and scan together
    int fused;          // that launch was asked for (GDN_FLAG_FUSED_LAUNCH)
    int ready_clear;    // the caller vouches that the ready flags are zero (GDN_FLAG_READY_FLAGS_CLEAR)
    int32_t* err;         // error latch in the workspace header: set when a scan workgroup of that launch gave up waiting
    int32_t* err_caller;  // the caller's own error word (gdn_args::error_word) or NULL
    uint32_t spin_limit;  // polls of a ready flag before giving up
    int no_producers;     // GDN_FLAG_DEBUG_NO_PRODUCERS
    uint64_t* cycle_out;  // measurement build (GDN_CYCLE_BUDGET) only: where sampled waves of the half-slice scan report; else NULL
    int rec16;          // the fragments of T diag(beta) and P are laid out for v_mfma_f32_16x16x32_bf16 (the half-slice scan)
    // left-padded batch: zeros at the padding of o (GDN_FLAG_ZERO_PADDING).  The last field: behind pad_lens it moved the kernel arguments
    // that follow, and the half-slice scan of 1024 chunks (32 chains, K = 128, V = 256) took 1310 us instead of 1245
    int zero_padding;
};

// The shapes the one-launch forward is used for: its scan workgroups (one per 64 columns of every chain, the chains rounded
// up to a multiple of 8) fill between 3/8 and 1/2 of the compute units.  With fewer chains the two-kernel path's scan, one
// slice per CU, is the faster one and prepare is short; with more, too few CUs are left for the producers.
// And the chains number at least 5/32 of the CUs (40 of 256).  Per chunk of a chain the one-launch scan (a pair of waves
// per slice, two slices per CU) is ~0.4 us slower than the half-slice scan of the two-kernel path, and what it saves is
// the prepare kernel, ~0.0115 us per chunk and chain: both grow with the sequence length, so the sign of the difference
// depends on the number of chains alone.  Measured at steady clocks: 64 chains (B = 4, H = 16, V = 128) 0.109 ms in one
// launch against 0.120 ms; 32 chains (H = 32, V = 256, T = 65536) 1.645 ms against 1.565 ms.
inline bool fused_launch_window(int64_t chains, int V, int num_cus) {
    const int64_t scan_wgs = (chains + 7) / 8 * 8 * (V / 64);
    return scan_wgs <= (int64_t)num_cus / 2 && scan_wgs >= (int64_t)num_cus * 3 / 8 && chains * 32 >= (int64_t)num_cus * 5;
}

// Kernel choice of the scan (plan_scan, gdn_chunk32.hip)
struct ScanPlan {
    int nw;             // 32-column slices per workgroup
    bool half;          // a slice is scanned by two waves of 16 columns (records in the 16x16x32 fragment order)
    bool split_keys;    // ... or: 16 columns to a workgroup, two waves with half of the keys each (gdn_chunk_scan_keys.hip)
    bool direct;        // four slices per workgroup: the compute waves store the output themselves
    bool staged_saves;  // a saving scan whose saves go through LDS and the store wave: only there bf16 saves exist
    bool no_output;     // the scan without output runs
};
// what a saving launch asks for (gdn_chunk_saves)
struct SaveRequest {
    bool no_output = false, has_state = true, has_vnew = true, state_bf16 = false, vnew_bf16 = false;
    int save_every = 1;
};
ScanPlan plan_scan(int K, int64_t chains, int T, int V, bool packed, bool save, int records_given, int num_cus, const SaveRequest& req);

struct RecordLayout {
    uint32_t off_p, off_qs, off_ks, off_cs, off_eg, bytes;
};

// Record of one (head, chunk), the same for every K and V: the 6 non-zero fragments of T diag(beta) (T = (I + A)^-1)
// at 0, the 6 non-zero fragments of P, then three vectors of 64 fp32 row scales - of q at off_qs
// (e^{gamma} scale / |q|), of k for the state update at off_ks (e^{gamma_C - gamma} / |k|), of k S0 at off_cs
// (e^{gamma} / |k|) - and e^{gamma_C}.  q, k and v themselves are read from the caller's tensors by the scan, which
// forms V~ = T diag(beta) (V - diag(cs) K S0) itself: the record depends neither on V nor on the key dim.
inline RecordLayout record_layout(int K, int V) {
    (void)K, (void)V;
    RecordLayout r;
    r.off_p = 6 * FRAG_BYTES;
    r.off_qs = r.off_p + 6 * FRAG_BYTES;
    r.off_ks = r.off_qs + C * 4;
    r.off_cs = r.off_ks + C * 4;
    r.off_eg = r.off_cs + C * 4;
    r.bytes = (r.off_eg + 4 + 255u) & ~255u;
    return r;
}

// Where chunk slot `slot` of the grid lives: sequence, chunk of it, first token, valid length (0 = unused slot).
struct ChunkCoord {
    int n, c;
    int64_t b, t0;
    int len;
};

__device__ __forceinline__ ChunkCoord no_chunk() {
    ChunkCoord cc;
    cc.n = 0, cc.c = 0, cc.b = 0, cc.t0 = 0, cc.len = 0;
    return cc;
}

// chunk `c` of packed sequence n, whose place in the prefix is cu0 .. cu1
__device__ __forceinline__ ChunkCoord packed_chunk(const ChunkParams& p, int n, int c, int cu0, int cu1) {
    ChunkCoord cc;
    cc.n = n, cc.c = c, cc.b = 0;
    const int t0 = min(max(cu0, 0), p.T), len = min(max(cu1, t0), p.T) - t0;  // as packed_bounds
    cc.t0 = (int64_t)t0 + (int64_t)c * C;
    cc.len = min(C, len - c * C);
    return cc;
}

// The chunk of a slot, looked up once per item of the prepare step, between an item and the loads of the next; slots past the last
// one (the item grid is rounded up) hold none.  Rows of a batch:
struct FindInRows {
    __device__ __forceinline__ FindInRows(const ChunkParams&, int) {}
    __device__ __forceinline__ ChunkCoord operator()(const ChunkParams& p, int slot) const {
        if (slot >= p.TC) return no_chunk();
        ChunkCoord cc;
        cc.n = slot / p.NT;
        const int c = slot - cc.n * p.NT;
        cc.b = cc.n, cc.c = c;
        // the last `len` tokens of the row (clamped: a malformed prefix must not send a load out of the row)
        const int len = p.pad_lens == nullptr ? p.T : min(max(p.pad_lens[cc.n + 1] - p.pad_lens[cc.n], 0), p.T);
        cc.t0 = (int64_t)(p.T - len) + (int64_t)c * C;
        cc.len = min(C, len - c * C);
        return cc;
    }
};
// Packed sequences.  Up to 63 of them keep their prefixes in the lanes of two registers, and a lookup is one comparison per lane; a
// search waits for one load per step, seven of them in a row at 11 sequences (prepare, 32768 tokens, 16 heads, K = 128, at steady
// clocks: 91 - 95 -> 84 - 88 us; 40 sequences 103 -> 98; in rows, 8 x 4096 tokens, 82 -> 81).  Those few every wave adds up for itself
// from the lengths, and one wave of the launch writes them down for the scan or the sweeps behind it (publish): a launch of its own in
// front (chunk_offsets_kernel, which gives the same values) cost about 2 us of a forward: 3 sequences, 1000 tokens, 16 heads, K = V =
// 128 25.2 -> 23.2 us, 5 of 2290 tokens, 3 heads, K = 256, V = 512 50.9 -> 48.6, 11 of 32768 tokens 248.6 -> 245.4.
__host__ __device__ inline bool offsets_in_prepare(int N) { return N < WAVE; }
struct FindPacked {
    int off = 0, cu = 0;

    __device__ __forceinline__ FindPacked(const ChunkParams& p, int lane) {
        if (!offsets_in_prepare(p.N)) return;
        cu = p.cu_seqlens[min(lane, p.N)];
        off = chunks(p, lane);
        // inclusive prefix sums, capped at the record slots at every addition (as chunk_offsets_kernel's), then exclusive ones
        off = min(off, p.TC);
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const int y = __shfl_up(off, d, WAVE);
            if (lane >= d) off = min(off + y, p.TC);
        }
        off = __shfl_up(off, 1, WAVE);
        if (lane == 0) off = 0;
    }
    __device__ __forceinline__ int chunks(const ChunkParams& p, int lane) const {  // of sequence `lane` (bounds as in packed_bounds)
        const int next = __shfl_down(cu, 1, WAVE);
        const int t0 = min(max(cu, 0), p.T), len = min(max(next, t0), p.T) - t0;
        return lane < p.N ? (len + C - 1) / C : 0;
    }
    // one wave: the offsets, and the sequences by decreasing number of chunks (ties by index)
    __device__ __forceinline__ void publish(const ChunkParams& p, int lane) const {
        const int mine = chunks(p, lane);
        int rank = 0;
        for (int m = 0; m < p.N; m++) {
            const int theirs = __builtin_amdgcn_readlane(mine, m);
            rank += (theirs > mine || (theirs == mine && m < lane)) ? 1 : 0;
        }
        if (lane <= p.N) p.chunk_off[lane] = off;
        if (lane < p.N) p.seq_order[rank] = lane;
    }
    __device__ __forceinline__ ChunkCoord operator()(const ChunkParams& p, int slot) const {
        if (slot >= p.TC) return no_chunk();
        if (offsets_in_prepare(p.N)) {
            // lanes N and up hold off[N]: bit N says that the slot lies past the last chunk, the bits below it how many sequences have begun
            const uint64_t begun = __builtin_amdgcn_ballot_w64(off <= slot);
            if (begun >> p.N & 1) return no_chunk();
            const int n = (int)__builtin_popcountll(begun) - 1;
            return packed_chunk(p, n, slot - __builtin_amdgcn_readlane(off, n), __builtin_amdgcn_readlane(cu, n), __builtin_amdgcn_readlane(cu, n + 1));
        }
        if (slot >= p.chunk_off[p.N]) return no_chunk();
        int lo = 0, hi = p.N;  // largest n with chunk_off[n] <= slot
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (p.chunk_off[mid] <= slot) lo = mid;
            else hi = mid;
        }
        return packed_chunk(p, lo, slot - p.chunk_off[lo], p.cu_seqlens[lo], p.cu_seqlens[lo + 1]);
    }
};

__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 pack8(f32x4 lo, f32x4 hi) {
    bf16x8 r;
    r[0] = (bf16_t)lo[0], r[1] = (bf16_t)lo[1], r[2] = (bf16_t)lo[2], r[3] = (bf16_t)lo[3];
    r[4] = (bf16_t)hi[0], r[5] = (bf16_t)hi[1], r[6] = (bf16_t)hi[2], r[7] = (bf16_t)hi[3];
    return r;
}

typedef __attribute__((ext_vector_type(16))) float f32x16;

// v_mfma_f32_32x32x16_bf16:  A[i = l%32][k = 8 (l/32) + 0..7]   B[k = 8 (l/32) + 0..7][j = l%32]
//                            D[i = 8 (r/4) + 4 (l/32) + r%4][j = l%32],  r = 0..15 the register index
__device__ __forceinline__ f32x16 mfma32_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

}  // namespace gdn
