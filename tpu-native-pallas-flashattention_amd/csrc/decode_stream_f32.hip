// Streaming decode (decode_stream.hpp): float32 head dims 64 and 128.
#include "decode_stream.hpp"

namespace pf {

int stream_blocks_f32(int head_dim, bool small, bool fine) {
  if (fine) return small ? stream::blocks_per_cu<float, 64, 2, 4, true>() : stream::blocks_per_cu<float, 64, 2, 16, true>();
  if (head_dim == 64)
    return small ? stream::blocks_per_cu<float, 64, 2, 4>() : stream::blocks_per_cu<float, 64, 2, 16>();
  return small ? stream::blocks_per_cu<float, 128, 2, 4>() : stream::blocks_per_cu<float, 128, 2, 16>();
}

hipError_t launch_stream_f32(const DecodeParams& p, bool paged, hipStream_t stream) {
  if (p.D == 64) return stream::launch_pg<float, 64>(p, paged, stream);
  if (p.D == 128) return stream::launch_pg<float, 128>(p, paged, stream);
  return hipErrorInvalidValue;
}

}  // namespace pf
