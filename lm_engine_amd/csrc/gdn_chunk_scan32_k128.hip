// The chunked forward's kernels for K = 128 (gdn_chunk_scan32.h).

#include "gdn_chunk_scan32.h"

namespace gdn {

template int launch32<128>(ChunkParams& p, hipStream_t stream, hipEvent_t* events, int num_cus);

}  // namespace gdn
