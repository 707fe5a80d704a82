// The chunked forward's kernels for K = 256 (gdn_chunk_scan32.h).

#include "gdn_chunk_scan32.h"

namespace gdn {

template int launch32<256>(ChunkParams& p, hipStream_t stream, hipEvent_t* events, int num_cus);

}  // namespace gdn
