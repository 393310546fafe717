// The rule by which a row may be expanded (perm_expand.hip says why its limits are these).
// It is applied in three places -- to a host matrix (plain_expand_row), to device matrices
// (plain_expand_kernel) and to the rows of a repeated task (choose_sweep) -- and the first
// two must agree on every matrix: the host launches the sweep for the form it expects the
// kernel to choose.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pqb {

constexpr double kPivotLargest = 0x1p20;    // no entry's component is larger (or not finite)
constexpr double kPivotSmallest = 0x1p-20;  // the expanded row's entries are not smaller than this
constexpr double kPivotSpread = 0x1p-16;    // nor than this of the matrix's largest

// Whole numbers of up to 21 bits times a power of two: the sum over all rows adds up small
// ones without rounding, which a division would lose.
constexpr int kGridBits = 20;

__host__ __device__ inline uint64_t double_bits(double v) {
    uint64_t b;
    __builtin_memcpy(&b, &v, sizeof(b));
    return b;
}

// Exponent of the lowest set bit of v (finite), larger than any for v = 0.
__host__ __device__ inline int lowest_bit(double v) {
    const uint64_t b = double_bits(v);
    const int e = (int)(b >> 52 & 0x7ff);
    const uint64_t m = (b & 0xfffffffffffffull) | (e ? 1ull << 52 : 0);
    return m ? (e ? e : 1) - 1075 + __builtin_ctzll(m) : 4096;
}

__host__ __device__ inline int lowest_bit(double re, double im) {
    const int x = lowest_bit(re), y = lowest_bit(im);
    return x < y ? x : y;
}

// Whether entries whose lowest bit is `low` and largest component `most` (at least
// kPivotSmallest, where it matters) lie off every such grid.
__host__ __device__ inline bool off_grid(int low, double most) {
    return low < (int)(double_bits(most) >> 52) - 1023 - kGridBits;
}

__host__ __device__ inline bool pivot_admits(double re, double im) {
    return __builtin_fabs(re) <= kPivotLargest && __builtin_fabs(im) <= kPivotLargest;
}

// Least magnitude (larger component) of the entries of a row that may be expanded.
__host__ __device__ inline double pivot_least(double most) {
    const double s = kPivotSpread * most;
    return s > kPivotSmallest ? s : kPivotSmallest;
}

}  // namespace pqb
