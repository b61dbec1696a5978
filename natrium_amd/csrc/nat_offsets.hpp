// Reach of the 32-bit byte offsets with which a kernel reads a direction and its opposite.
#pragma once
#include <cstdint>

namespace nat {

// A buffer resource that starts at the array of the lower of two opposite directions, `apart`
// arrays from the other one, is read up to the end of the other's array: apart + 1 arrays. Whether
// the offset of every byte of them, and of a 16-byte load at their end, stays below 2^32.
constexpr bool pair_offsets_fit(int64_t apart, int64_t stride, int64_t elem_bytes) {
  return (apart + 1) * stride * elem_bytes <= 0xfffffff0ll;
}

}  // namespace nat
