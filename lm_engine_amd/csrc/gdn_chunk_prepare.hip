// The prepare step of the chunked forward, and of the backward's sweeps, as a kernel of its own (gdn_chunk_prepare32.h).

#include "gdn_chunk32_common.h"
#include "gdn_chunk_prepare32.h"
#include "gdn_launch.h"

namespace gdn {

// ------------------------------------------------------------------------------------------
// persistent workgroups of four waves, three per CU
// ------------------------------------------------------------------------------------------
// SWEEP: the records of the backward's sweeps, and gamma, beta and the inverse norms per token (sw)
template <int K, bool SWEEP, typename Find>
__global__ __launch_bounds__(PREP_THREADS, (K > 128 ? 1 : 3)) void chunk_prepare32_kernel(const ChunkParams p, const SweepScalars sw) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[prepare32_lds_bytes<K>()];
    // Work items: (chunk slot, head), the slots rounded up to a multiple of 8.  Workgroup i runs on XCD i % 8 and
    // takes items i, i + grid, ... with the grid a multiple of 8, so w % 8 names the XCD.  That digit goes into
    // the slot number and the heads rotate with the rest: every XCD works on all heads.  The rows of one head
    // lie a whole token row (a multiple of 2 KiB) apart, so they fall on few channels of an XCD's L2; an XCD
    // that only ever sees one or two heads would send all its q, k, v traffic there.
    const uint32_t items = (uint32_t)((p.TC + 7) / 8) * 8u * (uint32_t)p.H;  // the launcher rejects more than 2^31
    if (blockIdx.x >= items) return;
    const uint32_t H = (uint32_t)p.H;
    auto item_of = [H](uint32_t w, int& h, int& slot) {
        const uint32_t j = w / 8u, jh = j / H;
        h = (int)(j - jh * H);
        slot = (int)(jh * 8u + w % 8u);
    };
    const uint32_t rounds = (items - blockIdx.x + gridDim.x - 1) / gridDim.x;
    if constexpr (std::is_same_v<Find, FindPacked>) {
        if (offsets_in_prepare(p.N) && blockIdx.x == gridDim.x - 1 && threadIdx.x < WAVE) Find(p, threadIdx.x).publish(p, threadIdx.x);
    }
    chunk_prepare32_body<K, 1, false, SWEEP, Find>(p, lds, item_of, items, blockIdx.x, gridDim.x, rounds, nullptr, 0, sw);
}

// workgroups of the prepare kernel: three per CU (LDS and registers allow it), a multiple of 8, see the kernel
static int prepare_grid(const ChunkParams& p, int num_cus) {
    const int64_t items = (int64_t)((p.TC + 7) / 8) * 8 * p.H;
    const int64_t cap = (int64_t)(3 * num_cus + 7) / 8 * 8;
    return items >= ((int64_t)1 << 31) ? 0 : (int)(items < cap ? items : cap);  // (the kernel counts items in 32 bits)
}

template <bool SWEEP, typename Find>
static int launch_prepare(const ChunkParams& p, const SweepScalars& sw, int K, hipStream_t stream, int num_cus) {
    const int grid = prepare_grid(p, num_cus);
    if (grid == 0) return GDN_ERR_UNSUPPORTED;
    if (K == 64) hipLaunchKernelGGL((chunk_prepare32_kernel<64, SWEEP, Find>), dim3(grid), dim3(PREP_THREADS), 0, stream, p, sw);
    else if (K == 128) hipLaunchKernelGGL((chunk_prepare32_kernel<128, SWEEP, Find>), dim3(grid), dim3(PREP_THREADS), 0, stream, p, sw);
    else if (K == 256) hipLaunchKernelGGL((chunk_prepare32_kernel<256, SWEEP, Find>), dim3(grid), dim3(PREP_THREADS), 0, stream, p, sw);
    else return GDN_ERR_UNSUPPORTED;
    return (int)hipGetLastError();
}

int launch_prepare32(const ChunkParams& p, int K, hipStream_t stream, int num_cus) {
    const SweepScalars none = {};
    return p.cu_seqlens != nullptr ? launch_prepare<false, FindPacked>(p, none, K, stream, num_cus) : launch_prepare<false, FindInRows>(p, none, K, stream, num_cus);
}

// the prepare step of the backward's sweeps
int launch_prepare_sweeps(ChunkParams& p, const SweepScalars& sw, int K, hipStream_t stream, int num_cus) {
    p.rec16 = 1;
    return p.cu_seqlens != nullptr ? launch_prepare<true, FindPacked>(p, sw, K, stream, num_cus) : launch_prepare<true, FindInRows>(p, sw, K, stream, num_cus);
}

}  // namespace gdn
