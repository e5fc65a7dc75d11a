// Runs of packed flags: the bytes that hold bits [lo, hi).  (constexpr: the same on host and device.)
#pragma once
#include <cstdint>

namespace fo {

struct FlagRange {
  uint32_t lo, hi;
  constexpr uint32_t first() const { return lo >> 3; }
  // (of an empty range the byte that its first bit would be in: in front of hi there may be no bit at all)
  constexpr uint32_t last() const { return (lo < hi ? hi - 1 : lo) >> 3; }
  // byte `at`, of value v, without the bits outside of the range
  constexpr uint32_t trim(uint32_t at, uint32_t v) const {
    if (at == lo >> 3) v &= 0xFFu << (lo & 7);
    if (at == hi >> 3) v &= (1u << (hi & 7)) - 1u;
    return at <= last() ? v : 0u;
  }
};

}  // namespace fo
