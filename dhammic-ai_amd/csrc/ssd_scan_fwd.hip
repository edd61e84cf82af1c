// Forward chunk scan entry of the general bf16 path, and the LDS size the host checks (both dtypes: it
// bounds the shapes the C ABI takes).
#include "ssd_scan_fwd_impl.h"

size_t lds_chunk_scan_fwd(int dtype, const SsdDims& d) {
  return lds_scan_fwd_hs(dtype == 1 ? 2 : 4, d, fwd_heads_per_block(dtype, d));
}
