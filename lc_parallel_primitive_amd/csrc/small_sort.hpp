// small_sort.hpp — one-workgroup radix sort of small inputs (small_sort.hip).
#pragma once

#include "common.hpp"

namespace lcpp {

// Most keys one workgroup sorts.
constexpr uint64_t small_sort_max(int key_bytes) { return key_bytes == 4 ? 16384 : 8192; }

// Sorts n <= small_sort_max(key_bytes) keys (4 or 8 bytes, `kind` as KeyKind in
// radix_sort.hip) in one launch; vals_in != NULL moves val_bytes-sized values
// with them.  `match`: rank by ballot match.  *status is zeroed.
int small_sort_launch(int key_bytes, int kind, bool descending, bool match, const void *keys_in, void *keys_out,
                      const void *vals_in, void *vals_out, int val_bytes, uint32_t n, uint32_t *status,
                      hipStream_t s);

}  // namespace lcpp
