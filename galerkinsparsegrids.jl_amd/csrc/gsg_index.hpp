// gsg_index.hpp -- quotients by multiplication (device code, and host code without HIP)
#pragma once
#include <cstdint>

namespace gsg {

// n / d for every 0 <= n < 2^31 as (n mul / 2^32) >> shift.  With 2^s < d < 2^(s + 1) and
// mul = ceil(2^(32 + s) / d), n mul / 2^(32 + s) is above n / d by less than n / 2^(32 + s),
// which is less than 1 / d as n d < 2^(32 + s): the floor is exact.  A power of two above 1
// takes mul = 2^31 and shifts the rest; d = 1 has no mul of 32 bits (the caller's case).
struct QuotMul {
  uint32_t mul, shift;
};
constexpr QuotMul quot_mul(uint32_t d) {
  uint32_t s = 0;
  while ((d >> s) > 1) ++s;
  if ((uint32_t(1) << s) == d) return d == 1 ? QuotMul{0, 0} : QuotMul{uint32_t(1) << 31, s - 1};
  return QuotMul{uint32_t(((uint64_t(1) << (32 + s)) + d - 1) / d), s};
}
constexpr uint32_t mul_hi(uint32_t a, uint32_t b) { return uint32_t((uint64_t(a) * b) >> 32); }
constexpr uint32_t quot(uint32_t n, QuotMul q) { return mul_hi(n, q.mul) >> q.shift; }

}  // namespace gsg
