// tie_repair.hpp — last step of the 8-byte key sorts that leave their low
// digits out (tie_repair.hip).
#pragma once

#include "small_sort.hpp"

namespace lcpp {

// Enqueues the repair of keys[0..n) (8-byte, `kind` a KeyKind) that are sorted,
// stably, by their sort keys' bits from *cut on: every run of keys equal in
// those bits is put in order by the others.  *cut == 0: nothing is done.  vals
// (val_bytes 4 or 8; NULL: none) move along; ktmp / vtmp are scratch of n
// elements.
int tie_repair_launch(int kind, bool descending, void *keys, void *vals, int val_bytes, void *ktmp, void *vtmp,
                      uint32_t n, const uint32_t *cut, hipStream_t s);

}  // namespace lcpp
