// Streaming decode (decode_stream.hpp): the 16-bit head_dim 128 kernels, the
// dispatch over element types and head dims, and the persistent grid size.
// Head dims 64 and 256 are built in decode_stream_dims.hip, float32 in
// decode_stream_f32.hip.
#include "decode_stream.hpp"

namespace pf {

// Supported forms. Rows of 64 or 128 elements (16-bit also 256), whole page
// groups (4 rows; 8 for 128-byte rows, where one load covers 8). Groups of
// more than 16 heads are cut into 16-head slices that each read the K/V, so
// off the 16-bit head_dim 128 path those stay with the generic kernel, which
// reads them once for 32 heads.
bool decode_stream_supported(int dtype, int head_dim, int group, bool paged, int page_size) {
  const bool f32 = dtype == kF32;
  if (head_dim != 64 && head_dim != 128 && (f32 || head_dim != 256)) return false;
  const bool wide_group_ok = !f32 && head_dim == 128;
  if (group > 16 && !wide_group_ok) return false;
  return !paged || page_size % (!f32 && head_dim == 64 ? 8 : 4) == 0;
}

int stream_blocks_dims(int head_dim, bool small);
int stream_blocks_f32(int head_dim, bool small, bool fine);
hipError_t launch_stream_dims(const DecodeParams& p, int dtype, bool paged, hipStream_t stream);
hipError_t launch_stream_f32(const DecodeParams& p, bool paged, hipStream_t stream);

// Resident one-wave workgroups of the streaming kernel on the current device
// (the persistent grid size). The device's CU count and the occupancy of
// every kernel variant are queried once per device (std::call_once) and
// cached; later calls cost one hipGetDevice. Without a usable device (a
// host-only query), MI355X's 256 CUs and the LDS-limited occupancy are
// assumed.
namespace {

constexpr int kMaxDevices = 64;
// variants: 16-bit head_dim 128 at 2, 3, 4 stages; 16-bit 64, 256; float32 64,
// 128; float32 64 with 16-key stages
constexpr int kVariants = 8;

struct StreamOccupancy {
  std::once_flag once;
  int cus = 0;
  int per_cu[kVariants][2] = {};  // [variant][query rows 4 / 16]
};
StreamOccupancy g_occupancy[kMaxDevices];

void query_occupancy(StreamOccupancy* o, int dev) {
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return;
  o->cus = cus;
  o->per_cu[0][0] = stream::blocks_per_cu<bf16_t, 128, 2, 4>();
  o->per_cu[0][1] = stream::blocks_per_cu<bf16_t, 128, 2, 16>();
  o->per_cu[1][0] = stream::blocks_per_cu<bf16_t, 128, 3, 4>();
  o->per_cu[1][1] = stream::blocks_per_cu<bf16_t, 128, 3, 16>();
  o->per_cu[2][0] = stream::blocks_per_cu<bf16_t, 128, 4, 4>();
  o->per_cu[2][1] = stream::blocks_per_cu<bf16_t, 128, 4, 16>();
  for (int s = 0; s < 2; ++s) {
    o->per_cu[3][s] = stream_blocks_dims(64, s == 0);
    o->per_cu[4][s] = stream_blocks_dims(256, s == 0);
    o->per_cu[5][s] = stream_blocks_f32(64, s == 0, false);
    o->per_cu[6][s] = stream_blocks_f32(128, s == 0, false);
    o->per_cu[7][s] = stream_blocks_f32(64, s == 0, true);
  }
}

}  // namespace

int decode_stream_waves(int dtype, int head_dim, int stages, int group, bool fine) {
  const bool f32 = dtype == kF32;
  const int sm = group <= 4 ? 0 : 1;
  const bool ring = !f32 && head_dim == 128;  // the variants with a tunable ring depth
  const int ns = ring && stages >= 2 && stages <= 4 ? stages : 2;
  const int v = fine ? 7 : ring ? ns - 2 : f32 ? (head_dim == 64 ? 5 : 6) : (head_dim == 64 ? 3 : 4);
  int per_cu = 0, cus = 0;
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices) {
    StreamOccupancy& o = g_occupancy[dev];
    std::call_once(o.once, query_occupancy, &o, dev);
    cus = o.cus;
    per_cu = o.per_cu[v][sm];
  }
  if (cus <= 0) cus = 256;
  if (per_cu <= 0) {
    using stream::StreamGeo;
    const int qr = sm == 0 ? 4 : 16;
    const int slot = fine                ? StreamGeo<float, 64, true>::slot_bytes(qr)
                     : f32 && head_dim == 64 ? StreamGeo<float, 64>::slot_bytes(qr)
                     : f32               ? StreamGeo<float, 128>::slot_bytes(qr)
                     : head_dim == 64    ? StreamGeo<bf16_t, 64>::slot_bytes(qr)
                     : head_dim == 128   ? StreamGeo<bf16_t, 128>::slot_bytes(qr)
                                         : StreamGeo<bf16_t, 256>::slot_bytes(qr);
    per_cu = 160 * 1024 / (ns * slot);
  }
  return cus * (per_cu > 1 ? per_cu : 1);
}

int decode_stream_qrows(int group) { return group <= 4 ? 4 : 16; }

hipError_t launch_decode_stream(const DecodeParams& p, int dtype, bool paged, hipStream_t stream) {
  if (dtype == kF32) return launch_stream_f32(p, paged, stream);
  if (p.D != 128) return launch_stream_dims(p, dtype, paged, stream);
  return dtype == kBF16 ? stream::launch_pg<bf16_t, 128>(p, paged, stream)
                        : stream::launch_pg<f16_t, 128>(p, paged, stream);
}

}  // namespace pf
