// Chunked forward of the gated delta rule (K = 64, 128, 256): the choice of the scan kernel and the dispatch over the key dim.  The
// kernels: gdn_chunk_scan32.h, a translation unit per key dim, and gdn_chunk_scan_keys.hip.

#include "gdn_chunk_common.h"
#include "gdn_launch.h"

namespace gdn {

template <int K>
int launch32(ChunkParams& p, hipStream_t stream, hipEvent_t* events, int num_cus);  // gdn_chunk_scan32_k*.hip
extern template int launch32<64>(ChunkParams& p, hipStream_t stream, hipEvent_t* events, int num_cus);
extern template int launch32<128>(ChunkParams& p, hipStream_t stream, hipEvent_t* events, int num_cus);
extern template int launch32<256>(ChunkParams& p, hipStream_t stream, hipEvent_t* events, int num_cus);

// Which scan kernel a launch gets: compute waves (32-column slices) per workgroup, and whether a slice is split over
// two half-slice waves.
ScanPlan plan_scan(int K, int64_t chains, int T, int V, bool packed, bool save, int records_given, int num_cus, const SaveRequest& req) {
    // Slices per scan workgroup: one while that gives no more workgroups than CUs, so that every slice has a CU's load
    // bandwidth to itself; otherwise 2 or 4 slices of a chain share the records through one workgroup's LDS (they must
    // divide the V / 32 tiles).
    const int vtiles = V / 32;
    int nw = 1;
    while (nw < 4 && vtiles % (2 * nw) == 0 && chains * (vtiles / nw) > (int64_t)num_cus) nw *= 2;
    // Packed batches are ragged as a rule, and their chains start longest first (chunk_offsets_kernel): the launch then
    // takes as long as the longest chain, which runs faster the fewer slices share its workgroup, while the workgroups
    // that do not fit at first fill in behind the short chains.  So up to two workgroups per CU are accepted there.
    // (Configuration 2, 11 sequences of 202 .. 6350 tokens, H = 16: 246 us with four slices per workgroup, 193 us with two.)
    if (packed && !save && nw > 1 && chains * (vtiles / (nw / 2)) <= 2 * (int64_t)num_cus) nw /= 2;
    if (save && nw == 2) nw = 1;  // the saving variant exists for 1 and 4 slices per workgroup
    // The saving scan of a packed batch: started longest first as well, its half-slice variant, whose saves go through LDS,
    // finishes a ragged batch sooner than four slices per workgroup storing from their compute waves (11 sequences of 202 .. 6350
    // tokens, H = 16, 2.75 workgroups per CU: 352 us against 575 us).
    if (save && packed && !records_given && K <= 128) nw = 1;
    if (K > 128) nw = 1;  // K = 256 scans on half slices, also as the saving variant and on given records, or with the keys split (below)
    if (records_given == 2) nw = 1;  // records given in the half-slice scan's fragment order
    ScanPlan plan;
    plan.nw = nw;
    // a slice with a CU to itself is scanned by two waves of 16 columns each; the records are laid out for them
    plan.half = K > 128 || records_given == 2 || (nw == 1 && !records_given);
    // K = 256, and twice as many workgroups still have a CU each: 16 columns to a workgroup and the keys over two waves, whose chunk step is a
    // sixth shorter.  Forward, half slices | this, V = 512: 4 x 777 tokens, 2 heads, 256 workgroups 36.2 | 33.3 us, 4 x 64 14.5 | 14.5, 2000
    // tokens 68.7 | 60.3.  More workgroups would run in rounds.
    plan.split_keys = plan.half && !save && K == 256 && (chains + 7) / 8 * 8 * (V / 16) <= (int64_t)num_cus;
    // Four slices to a workgroup, rows of two to four chunks: what goes through LDS is stored a chunk later, with nothing left to compute beside
    // it, and a short last chunk leaves the memory idle before.  Through LDS | from the compute waves, 16 heads, K = V = 128: 20 x 65 tokens 31.7 |
    // 30.4 us, 20 x 160 43.1 | 41.0, 40 x 200 76.2 | 75.2, 100 x 65 105 | 100, 100 x 90 110 | 106, K = 64, 40 x 65 39.6 | 38.4.  The loaders
    // are better where the chunks are full or many workgroups' stores crowd each other: 20 x 256 50.1 | 49.9, 40 x 256 79.0 | 79.5, 100 x 127 120 |
    // 123, 100 x 200 177 | 182, K = 64, 100 x 127 89.4 | 90.5, 40 x 200 57.5 | 59.4; and with one chunk, 20 x 64 25.4 | 25.6.
    plan.direct = nw == 4 && !save && !packed && T > C && (T <= 2 * C - C / 4 || (K == 128 && T < 4 * C && chains * (vtiles / nw) <= 3 * (int64_t)num_cus));
    // Saves go through LDS and the store wave in the half-slice scan: always at K <= 128; at K = 256 only in the scan
    // without output (no rows of q in LDS), with bf16 V~, and fp32 states at every second chunk at most (one buffer).
    plan.staged_saves = save && plan.half &&
                        (K <= 128 || (req.no_output && (!req.has_vnew || req.vnew_bf16) && (!req.has_state || req.state_bf16 || req.save_every >= 2)));
    plan.no_output = plan.staged_saves && req.no_output && K >= 128;
    return plan;
}

int launch_chunk32(ChunkParams& p, int K, hipStream_t stream, hipEvent_t* events, int num_cus) {
    if (K == 64) return launch32<64>(p, stream, events, num_cus);
    if (K == 128) return launch32<128>(p, stream, events, num_cus);
    if (K == 256) return launch32<256>(p, stream, events, num_cus);
    return GDN_ERR_UNSUPPORTED;
}

}  // namespace gdn
