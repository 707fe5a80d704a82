// Records and parameters of the backward's two sweeps (gdn_chunk_sweep.hip), shared with the prepare step that writes the
// records (gdn_chunk_prepare32.h) and the host side (gdn_chunk.hip).
#pragma once

#include "gdn_chunk_common.h"

namespace gdn {

// Record of one (head, chunk) for the sweeps, fragments in the lane order of the 16x16x32 MFMA: what the forward sweep reads (six
// fragments of T diag(beta), four vectors of 64 fp32: ks | cs | e^{gamma_C} in every entry | not used), then what the reverse sweep
// reads (six fragments of T^T, six of P^T, qs | ks | -beta cs | e^{gamma_C} in every entry).  Scales as in gdn_chunk_sweep.hip; those
// of rows past the end of a short chunk are zero.
constexpr uint32_t SWEEP_REC_FWD = 0, SWEEP_REC_FWD_SCALES = SWEEP_REC_FWD + 6 * FRAG_BYTES;
constexpr uint32_t SWEEP_REC_REV = SWEEP_REC_FWD_SCALES + 4 * C * 4, SWEEP_REC_REV_P = SWEEP_REC_REV + 6 * FRAG_BYTES;
constexpr uint32_t SWEEP_REC_REV_SCALES = SWEEP_REC_REV_P + 6 * FRAG_BYTES;
constexpr uint32_t SWEEP_RECORD_BYTES = SWEEP_REC_REV_SCALES + 4 * C * 4;

struct SweepParams {
    const bf16_t* q;
    const bf16_t* k;
    const bf16_t* v;  // forward: v; reverse: dO
    int64_t q_stride_b, q_stride_t, q_stride_h;
    int64_t k_stride_b, k_stride_t, k_stride_h;
    int64_t v_stride_b, v_stride_t, v_stride_h;
    const uint8_t* rec;  // [H][TC]
    uint32_t rec_bytes;
    const float* s_in;  // [N][H][K][V]: initial state, or gradient of the final state (NULL: zeros)
    float* s_out;       // gradient of the initial state (reverse), or NULL
    bf16_t* save_state; // [N H][save_nc][V / 32][K][32]
    bf16_t* save_v;     // [N H][save_nc][V / 32][64][32]
    int save_nc;
    const int32_t* cu_seqlens;  // packed sequences, else NULL
    const int32_t* pad_lens;    // left-padded batch: prefix sums of the valid lengths, else NULL
    const int32_t* chunk_off;   // packed: [N + 1], [N] as in ChunkParams
    const int32_t* seq_order;
    int T, H, V, N, NT, TC, qk_div;
};

// What the prepare step writes beside the sweeps' records, for the chunk-local kernel: [N H][nc][64] each
struct SweepScalars {
    float* gamma;
    float* beta;
    float* rq;
    float* rk;
    int nc;
};

}  // namespace gdn
