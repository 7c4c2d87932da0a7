// Division by divisors that the host knows.
#pragma once
#include <stdint.h>

namespace vsp {

// Division of 0 <= n < 2^31 by a divisor the host knows: a high multiply, an add and a shift instead of the forty-odd instructions (a reciprocal and
// its corrections, 0.1 to 0.2 us of a kernel's first microsecond) of an integer division.  Granlund and Montgomery, "Division by invariant integers
// using multiplication", 1994: with s = ceil(log2 d) and m = floor(2^32 (2^s - d) / d) + 1, n / d = (mulhi(m, n) + n) >> s.
struct FastDiv {
    uint32_t d, m, s;
    static FastDiv of(int64_t divisor) {
        FastDiv f{divisor > 0 ? (uint32_t)divisor : 1u, 0, 0};
        while (((uint64_t)1 << f.s) < f.d) ++f.s;
        f.m = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << f.s) - f.d)) / f.d + 1);
        return f;
    }
    __host__ __device__ uint32_t div(uint32_t n) const { return ((uint32_t)(((uint64_t)m * n) >> 32) + n) >> s; }
    __host__ __device__ uint32_t mod(uint32_t n, uint32_t quotient) const { return n - quotient * d; }
};

}  // namespace vsp
