// The decode attention kernels of 32-bit float caches.
#include "decode_attn_kernels.h"

namespace wnw {
template hipError_t launch_attn_d<float>(int, int64_t, const AttnParams&, int64_t, hipStream_t);
}  // namespace wnw
