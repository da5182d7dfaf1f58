// tq_attention_k4_pq.hip -- the fused decode kernels for 4-bit
// PQ (standard codebook in bits-wide slots) records: every head_dim, head-group and
// workgroup shape, with the inline split-K merge and for the reference
// ABI's separate merge launch.  One unit per bit width and cache mode, so
// that the kernels build in parallel.
#include "tq_decode_kernel.h"

namespace tqa {
template void launch_stream_bm<4, kModePq, true>(AttnArgs &, int, int, dim3, hipStream_t, tqh::AppendToken *);
template void launch_stream_bm<4, kModePq, false>(AttnArgs &, int, int, dim3, hipStream_t, tqh::AppendToken *);
}  // namespace tqa
