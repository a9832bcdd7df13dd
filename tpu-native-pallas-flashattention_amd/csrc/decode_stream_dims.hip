// Streaming decode (decode_stream.hpp): 16-bit head dims 64 and 256.
#include "decode_stream.hpp"

namespace pf {

int stream_blocks_dims(int head_dim, bool small) {
  if (head_dim == 64)
    return small ? stream::blocks_per_cu<bf16_t, 64, 2, 4>() : stream::blocks_per_cu<bf16_t, 64, 2, 16>();
  return small ? stream::blocks_per_cu<bf16_t, 256, 2, 4>() : stream::blocks_per_cu<bf16_t, 256, 2, 16>();
}

hipError_t launch_stream_dims(const DecodeParams& p, int dtype, bool paged, hipStream_t stream) {
  if (p.D == 64)
    return dtype == kBF16 ? stream::launch_pg<bf16_t, 64>(p, paged, stream)
                          : stream::launch_pg<f16_t, 64>(p, paged, stream);
  if (p.D == 256)
    return dtype == kBF16 ? stream::launch_pg<bf16_t, 256>(p, paged, stream)
                          : stream::launch_pg<f16_t, 256>(p, paged, stream);
  return hipErrorInvalidValue;
}

}  // namespace pf
