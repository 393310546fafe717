// Which integer matrices the exact sweep on the FP64 pipe (perm_exact.hip) takes.  Host
// only and free of HIP, so that the rule can be checked by itself over its whole range.
#pragma once

#include <algorithm>
#include <cstdint>

namespace pqb {

// Steps between flushes for a matrix of C columns whose column abs sums are at most
// cmax >= 0; 0: its products of ceil(C / 3) column sums may exceed 46 bits.
inline int exact_fp64_flush(int64_t cmax, int C) {
    constexpr int64_t kMost = (int64_t)1 << 46;
    const int64_t c = std::max<int64_t>(cmax, 1);
    int64_t q = 1;
    for (int k = 0; k < (C + 2) / 3; ++k) {
        if (q > kMost / c) return 0;  // before the product, which may not fit 64 bits
        q *= c;
    }
    int e = 0;
    while (((int64_t)1 << e) < q) ++e;
    return 1 << std::min(8, 140 - 3 * e);
}

}  // namespace pqb
