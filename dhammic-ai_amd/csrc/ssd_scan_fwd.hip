// The LDS size of the general bf16 forward chunk scan (ssd_scan_fwd_bf16.hip), for the host's check.
#include "ssd_scan_fwd_impl.h"

size_t lds_chunk_scan_fwd(const SsdDims& d) {
  return lds_scan_fwd_hs(sizeof(bf16), d, fwd_heads_per_block(sizeof(bf16), d));
}
