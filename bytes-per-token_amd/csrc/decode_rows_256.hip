// Many-row paged attention (decode_rows.h) in tiles of 256 rows.
#include "decode_rows.h"

namespace bpt {

hipError_t launch_rows_256(const DecodeParams& p, int kv_dtype, int scale_kind, hipStream_t stream, const LaunchEvents& ev) {
  return launch_rows_cfg<8, 8, 2>(p, kv_dtype, scale_kind, stream, ev);
}

}  // namespace bpt
