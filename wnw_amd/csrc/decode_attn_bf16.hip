// The decode attention kernels of bfloat16 caches.
#include "decode_attn_kernels.h"

namespace wnw {
template hipError_t launch_attn_d<bf16_t>(int, int64_t, const AttnParams&, int64_t, hipStream_t);
}  // namespace wnw
