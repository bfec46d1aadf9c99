// small_sort.hpp — one-workgroup radix sort of small inputs (small_sort.hip)
// and the key masks that it shares with radix_sort.hip.
#pragma once

#include "common.hpp"

namespace lcpp {

enum KeyKind { kUnsigned = 0, kSigned = 1, kFloat = 2 };

// Raw key -> sort key and back with masks: in(k) = k ^ (negative ? neg : pos) ^
// flip (the twiddles of common/util_type.h:98-175; flip inverts for descending
// order).  ZEROS (floating keys): `mz`, the sort key of -0.0, ranks as `pz`,
// that of +0.0.
template <class UK_, bool ZEROS>
struct KeyCode {
    using UK = UK_;
    UK neg, pos, flip, mz, pz;
    static constexpr UK kHigh = UK(1) << (sizeof(UK) * 8 - 1);
    static KeyCode of(int kind, bool desc)
    {
        const UK flip = desc ? UK(~UK(0)) : UK(0);
        return {kind == kFloat ? UK(~UK(0)) : kind == kSigned ? kHigh : UK(0), kind == kUnsigned ? UK(0) : kHigh, flip,
                UK(UK(~kHigh) ^ flip), UK(kHigh ^ flip)};
    }
    __device__ __forceinline__ UK in(UK k) const { return k ^ ((k & kHigh) ? neg : pos) ^ flip; }
    __device__ __forceinline__ UK out(UK t) const
    {
        const UK u = t ^ flip;
        return u ^ ((u & kHigh) ? pos : neg);
    }
    __device__ __forceinline__ UK ranked(UK t) const { return ZEROS && t == mz ? pz : t; }
    __device__ __forceinline__ uint32_t digit(UK t, uint32_t shift) const { return (uint32_t)(ranked(t) >> shift) & 255u; }
};

// Most keys one workgroup sorts.
constexpr uint64_t small_sort_max(int key_bytes) { return key_bytes == 4 ? 16384 : 8192; }

// Sorts n <= small_sort_max(key_bytes) keys (4 or 8 bytes, `kind` a KeyKind) in one launch; vals_in != NULL moves val_bytes-sized values
// with them.  `match`: rank by ballot match.  *status is zeroed.
int small_sort_launch(int key_bytes, int kind, bool descending, bool match, const void *keys_in, void *keys_out,
                      const void *vals_in, void *vals_out, int val_bytes, uint32_t n, uint32_t *status,
                      hipStream_t s);

}  // namespace lcpp
